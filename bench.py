#!/usr/bin/env python3
"""Decode throughput of RAMforge's hot path on one MI355X.

Workload (BASELINE.json metric): random-init Llama-3-8B-shape model (32
layers, d 4096, 32/8 heads, FFN 14336, vocab 128256), Q8_0 weights resident in
HBM, greedy decode.  One step = one token: output norm + logits matvec,
on-device argmax, embedding of the chosen token, 32 transformer layers.  The
prompt (32 random token ids) is forwarded before the timed region (batched,
rf_model_prefill).  Also measured, outside the decode line's value: the
prompt forwarded token by token (the reference's loop) against the batched
prefill, and a 512-token batched prompt.

Prints one JSON line with the decode tok/s, the roofline of the dominant
kernel (ffn RMSNorm + gate/up Q8_0 matvec + SiLU*up, timed with HIP events on
the stream it runs on), the Q8_0 4096x4096 matvec HBM GB/s
and the CPU baseline: the oracle restatement of the reference CPU path
(reference threading policy: Q8_0 matvecs single-threaded) timed on this
host on a bounded sample of the same workload.
"""
from __future__ import annotations

import argparse
import json
import os
import statistics
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

PEAK_HBM_GBS = 8000.0
PEAK_BF16_TFLOPS = 2500.0  # dense bf16 MFMA
METRIC = "decode tok/s (8B-shape Q8_0, 1 GPU); matvec achieved HBM GB/s vs peak"


def log(msg: str) -> None:
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def cpu_model_name() -> str:
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def matvec_q8_0_gbs(ctx, rf, syn, iters: int = 120):
    """Q8_0 4096x4096 matvec; weights rotate through ~1 GiB
    of distinct copies so the 256 MiB Infinity Cache cannot serve them."""
    out_dim = in_dim = 4096
    nblk = out_dim * in_dim // 32
    wbytes = nblk * 34
    copies = max(2, (1 << 30) // wbytes + 1)
    ws = []
    for i in range(copies):
        w = ctx.empty((wbytes,), "uint8", charge=f"bench:q8_0_4096:{i}")
        ctx.synth_blocks(syn.Q8_0, 1001, 0, nblk, 0.02 / 127, w)
        ws.append(w)
    import numpy as np

    x = ctx.array(np.random.default_rng(1).normal(0, 1, in_dim).astype(np.float32), "bench:q8_0_4096:x")
    y = ctx.empty((out_dim,), charge="bench:q8_0_4096:y")

    def per_call_ms():
        for i in range(copies):  # warm-up; with the repack cache on, packs each copy
            rf.matvec(ctx, syn.Q8_0, ws[i], (out_dim, in_dim), x, y)
        ctx.synchronize()
        e0, e1 = ctx.event(), ctx.event()
        ctx.record(e0, ctx.compute_stream)
        for i in range(iters):
            rf.matvec(ctx, syn.Q8_0, ws[i % copies], (out_dim, in_dim), x, y, stream=ctx.compute_stream)
        ctx.record(e1, ctx.compute_stream)
        ms = ctx.elapsed_ms(e0, e1) / iters
        ctx.destroy_event(e0)
        ctx.destroy_event(e1)
        return ms

    ms = per_call_ms()
    ctx.matvec_cache(copies * wbytes)
    ms_cached = per_call_ms()
    ctx.matvec_cache(0)
    alg = wbytes + 4 * in_dim + 4 * out_dim
    for a in ws + [x, y]:
        a.free()
    return {"config": "Q8_0 4096x4096 y=Wx, weights rotated over %d copies (%.2f GiB)" % (copies,
                                                                                      copies * wbytes / 2 ** 30),
            "us_per_call": round(ms * 1e3, 3), "algorithmic_bytes": alg,
            "achieved_GBs": round(alg / (ms * 1e-3) / 1e9, 1), "frac_of_peak": round(alg / (ms * 1e-3) / 1e9 /
                                                                                      PEAK_HBM_GBS, 4),
            "repack_cache": {"us_per_call": round(ms_cached * 1e3, 3),
                             "frac_of_peak": round(alg / (ms_cached * 1e-3) / 1e9 / PEAK_HBM_GBS, 4),
                             "note": "the same eager rf_matvec calls with rf_matvec_cache on (packed once, "
                                     "the packed kernel after)"}}


def host_cores() -> dict:
    try:
        usable = len(os.sched_getaffinity(0))
    except (AttributeError, OSError):
        usable = os.cpu_count() or 1
    return {"nproc": usable, "logical_cpus": os.cpu_count(), "model": cpu_model_name()}


def cpu_baseline(cfg, specs, first_token: int, steps: int):
    """Time the oracle (reference CPU path restated in C, reference threading
    policy: Q8_0 matvecs single-threaded, compute_dispatch.rs:219-254) on the
    same model: the prompt's first token forwarded at position 0, then `steps`
    greedy steps (logits, first-max argmax, forward), the first one untimed
    (warmup).  Returns the timing and the greedy tokens, which the GPU
    reproduces from the same start."""
    import oracle as orc

    t0 = time.perf_counter()
    T = orc.model_tensors(specs)
    gen_s = time.perf_counter() - t0
    m = orc.Model(cfg, T, kv_capacity=steps + 2, threads=1, use_simd=True)
    h = m.forward(first_token, 0)
    per, toks = [], []
    for i in range(steps):
        t0 = time.perf_counter()
        tok = orc.argmax(m.logits(h))
        h = m.forward(tok, i + 1)
        per.append(time.perf_counter() - t0)
        toks.append(tok)
        log(f"cpu step {i}{' (warmup)' if i == 0 else ''}: {per[-1]:.2f} s, token {tok}")
    m.close()
    timed = per[1:]
    med = statistics.median(timed)
    return {"value": round(1.0 / med, 5), "unit": "tok/s", "cores": 1, "kind": "port",
            "sample": (f"{len(timed)} greedy decode steps (logits + argmax + forward) of the same 8B-shape Q8_0 "
                       f"model after 1 warmup step, from the prompt's first token at position 0, median; oracle "
                       f"restatement of the reference CPU path, Q8_0 matvecs single-threaded as in "
                       f"compute_dispatch.rs:219-254; weights generated in {gen_s:.1f} s, untimed"),
            "host": host_cores(), "seconds_per_step": [round(p, 3) for p in timed]}, toks


def context_decode(ctx, m, cfg, n: int, steps: int, graph: bool) -> dict:
    """Decode tok/s at about n positions of context: n - 1 random prompt
    tokens forwarded by the batched prefill, then `steps` timed decode steps
    (after 4 untimed ones that capture the step graph of that context's
    attention regime)."""
    import numpy as np

    m.reset()
    toks = [int(t) for t in np.random.default_rng(n).integers(0, cfg["vocab_size"], n - 1)]
    t0 = time.perf_counter()
    m.prefill(toks)
    ctx.synchronize()
    pre_s = time.perf_counter() - t0
    m.use_graph(graph)
    m.decode_steps(4)
    ctx.synchronize()
    t0 = time.perf_counter()
    m.decode_steps(steps)
    ctx.synchronize()
    wall = time.perf_counter() - t0
    kv = 2 * 4 * cfg["block_count"] * cfg["head_count_kv"] * cfg["head_dim"] * (n + 4 + steps // 2)
    out = {"tok_s": round(steps / wall, 2), "ms_per_step": round(wall * 1e3 / steps, 4), "steps": steps,
           "positions": [n + 3, n + 3 + steps], "kv_bytes_per_step": kv, "prefill_s": round(pre_s, 3)}
    log(f"decode at context {n}: {out['tok_s']} tok/s ({out['ms_per_step']} ms/step; prompt of {n - 1} tokens "
        f"prefilled in {pre_s:.2f} s)")
    return out


def dominant_kernel(m) -> str:
    """Kernel instance that runs the ffn RMSNorm + gate/up + SiLU*up group of
    the 8B Q8_0 model, as the rocprofv3 kernel trace names it (the library
    reports the instance its launcher picks)."""
    return m.kernel_name("gateup") or "matvec_stream<Q8_0, EPI_SWIGLU> (GGUF layout)"


def under_tracer() -> bool:
    """True when this process runs under rocprofv3 (it exports its settings
    as ROCPROF_* / ROCPROFILER_* variables to the profiled program)."""
    return any(k.startswith(("ROCPROF_", "ROCPROFILER_")) for k in os.environ)


def trace_mean_us(kernel: str):
    """Mean duration of `kernel` in the committed kernel trace of the decode
    step (profiles/decode_8b_q8_0_kernel_stats.json), or None when the
    committed trace does not hold that exact kernel."""
    path = os.path.join(ROOT, "profiles", "decode_8b_q8_0_kernel_stats.json")
    try:
        tj = json.load(open(path))
    except (OSError, ValueError):
        return None
    row = tj.get("kernels", {}).get(kernel)
    return None if row is None else row.get("mean_us")



COPY_BYTES = 256 << 20


def traffic_probe(ctx, m, cfg, rf) -> int:
    """Launch only what the HBM-traffic counters are read for: one forward
    (so activations are defined), then the gate/up group of every layer once,
    then four plain device copies of COPY_BYTES (the calibration kernel)."""
    m.forward(1, 0)
    ctx.synchronize()
    ms, b, n = m.time_kernel("gateup", 1)
    src = ctx.empty((COPY_BYTES,), "uint8", charge="probe:copy:src")
    dst = ctx.empty((COPY_BYTES,), "uint8", charge="probe:copy:dst")
    for _ in range(4):
        ctx.copy(dst, src, COPY_BYTES)
    ctx.synchronize()
    print(json.dumps({"probe": "gateup", "kernel": dominant_kernel(m), "launches": n, "algorithmic_bytes": b,
                      "copy_bytes": COPY_BYTES, "copies": 4, "layers": cfg["block_count"]}), flush=True)
    src.free()
    dst.free()
    m.close()
    ctx.close()
    return 0


def attention_probe(rf, L: int, copies: int = 4) -> int:
    """Launch only what the attention counters are read for: RoPE + split-K
    attention + merge (32 q / 8 KV heads, hd 128, L positions; BASELINE config
    3) once on each of `copies` distinct K/V copies, then four plain device
    copies of COPY_BYTES (the calibration kernel for FETCH_SIZE/WRITE_SIZE)."""
    import numpy as np

    ctx = rf.Context(0)
    rng = np.random.default_rng(7)
    qh, kvh, hd, hist = 32, 8, 128, L - 1
    kv = [(ctx.array(rng.normal(0, 1, hist * kvh * hd).astype(np.float32)),
           ctx.array(rng.normal(0, 1, hist * kvh * hd).astype(np.float32))) for _ in range(copies)]
    q = ctx.array(rng.normal(0, 1, qh * hd).astype(np.float32))
    kc = ctx.array(rng.normal(0, 1, kvh * hd).astype(np.float32))
    vc = ctx.array(rng.normal(0, 1, kvh * hd).astype(np.float32))
    o = ctx.empty((qh * hd,))
    ctx.reserve(attention_bytes=ctx.attention_workspace_bytes(L, qh, kvh, hd), fixed=True)
    for kh, vh in kv:
        rf.apply_rope(ctx, q, kc, hist, hd, qh, kvh, 10000.0)
        rf.attention_checked(ctx, q, kh, vh, kc, vc, hist, qh, kvh, hd, out=o)
    src = ctx.empty((COPY_BYTES,), "uint8")
    dst = ctx.empty((COPY_BYTES,), "uint8")
    for _ in range(4):
        ctx.copy(dst, src, COPY_BYTES)
    ctx.synchronize()
    print(json.dumps({"probe": "attention", "positions": L, "launches": copies,
                      "algorithmic_bytes": 2 * L * kvh * hd * 4 + 2 * qh * hd * 4, "copy_bytes": COPY_BYTES,
                      "copies": 4}), flush=True)
    ctx.close()
    return 0


def matvec_probe(rf, spec: str, copies: int = 4) -> int:
    """Launch only what the matvec counters are read for: the GGUF-layout and
    the packed matvec of one shape ("Q4_0,14336,4096": type, out, in) once on
    each of `copies` distinct weight copies, then four plain device copies of
    COPY_BYTES (the calibration kernel for FETCH_SIZE / WRITE_SIZE)."""
    import numpy as np

    tn, out_dim, in_dim = spec.split(",")
    t = getattr(rf.GGML, tn)
    out_dim, in_dim = int(out_dim), int(in_dim)
    ctx = rf.Context(0)
    qk, bs = rf.BLOCK_GEOMETRY[t]
    nblk = out_dim * in_dim // qk
    wbytes = nblk * bs
    ws, ps = [], []
    for i in range(copies):
        w = ctx.empty((wbytes,), "uint8")
        ctx.synth_blocks(t, 7000 + i, 0, nblk, 0.02, w)
        p = ctx.empty((wbytes,), "uint8")
        rf.pack_weights(ctx, t, w, out_dim, in_dim, p)
        ws.append(w)
        ps.append(p)
    x = ctx.array(np.random.default_rng(3).normal(0, 1, in_dim).astype(np.float32))
    y = ctx.empty((out_dim,))
    for w in ws:
        rf.matvec(ctx, t, w, (out_dim, in_dim), x, y)
    for p in ps:
        rf.matvec_packed(ctx, t, p, (out_dim, in_dim), x, y)
    src = ctx.empty((COPY_BYTES,), "uint8")
    dst = ctx.empty((COPY_BYTES,), "uint8")
    for _ in range(4):
        ctx.copy(dst, src, COPY_BYTES)
    ctx.synchronize()
    print(json.dumps({"probe": "matvec", "type": tn, "shape": [out_dim, in_dim], "launches": copies,
                      "algorithmic_bytes": wbytes + 4 * in_dim + 4 * out_dim, "copy_bytes": COPY_BYTES,
                      "copies": 4}), flush=True)
    ctx.close()
    return 0


def kernel_bench(rf, syn, use_graph: bool, reps: int = 3) -> list:
    """BASELINE configs 1-3 at kernel level: each call rotates over distinct
    weight (or K/V) copies totalling >= 1.2 GiB so the 256 MiB Infinity Cache
    cannot serve them; the calls are captured into one hipGraph and replayed
    (GPU time incl. the graph's per-kernel launch cost), or issued eagerly
    for profiler runs (use_graph False: host-bound timings, use the trace)."""
    import numpy as np

    ctx = rf.Context(0)
    rng = np.random.default_rng(7)
    out = []

    def timed(calls, n_calls):
        for c in calls[:2]:  # warm every lazily created workspace outside capture
            c()
        ctx.synchronize()
        if use_graph:
            with ctx.capture() as cap:
                for c in calls:
                    c()
            g = cap.graph
            g.replay(1)
            ms = g.replay(reps) / n_calls
            g.close()
            return ms
        e0, e1 = ctx.event(), ctx.event()
        ctx.record(e0, ctx.compute_stream)
        for _ in range(reps):
            for c in calls:
                c()
        ctx.record(e1, ctx.compute_stream)
        return ctx.elapsed_ms(e0, e1) / (reps * n_calls)

    def record(config, kernel, ms, nbytes):
        gbs = nbytes / (ms * 1e-3) / 1e9
        out.append({"config": config, "kernel": kernel, "us": round(ms * 1e3, 3), "algorithmic_bytes": nbytes,
                    "GBs": round(gbs, 1), "frac_of_peak": round(gbs / PEAK_HBM_GBS, 4)})
        log(f"{config:34s} {kernel:28s} {ms * 1e3:8.2f} us {gbs:7.0f} GB/s")

    G = rf.GGML
    mats = [("Q8_0 4096x4096", G.Q8_0, 4096, 4096, 0.02 / 127), ("F32 4096x4096", G.F32, 4096, 4096, 1.0)]
    for t, tn in ((G.Q4_0, "Q4_0"), (G.Q4_K, "Q4_K"), (G.Q6_K, "Q6_K")):
        mats += [(f"{tn} 14336x4096", t, 14336, 4096, 0.02), (f"{tn} 4096x14336", t, 4096, 14336, 0.02)]
    # large single matrices (not BASELINE configs): a 70B-shape FFN matrix and the
    # Q6_K output projection of an 8B Q4_K_M model
    mats += [("Q8_0 28672x8192 (70B ffn)", G.Q8_0, 28672, 8192, 0.02 / 127),
             ("Q6_K 128256x4096 (8B output)", G.Q6_K, 128256, 4096, 0.02)]
    for name, t, out_dim, in_dim, mul in mats:
        qk, bs = rf.BLOCK_GEOMETRY[t]
        nblk = out_dim * in_dim // qk
        wbytes = nblk * bs
        copies = max(2, -(-(int(1.2 * 2 ** 30)) // wbytes))
        ws = []
        for i in range(copies):
            w = ctx.empty((wbytes,), "uint8", charge=f"kbench:{name}:{i}")
            ctx.synth_blocks(t, 5000 + i, 0, nblk, mul, w)
            ws.append(w)
        x = ctx.array(rng.normal(0, 1, in_dim).astype(np.float32), f"kbench:{name}:x")
        y = ctx.empty((out_dim,), charge=f"kbench:{name}:y")
        alg = wbytes + 4 * in_dim + 4 * out_dim
        calls = [lambda w=w: rf.matvec(ctx, t, w, (out_dim, in_dim), x, y) for w in ws]
        record(name, "matvec (GGUF layout)", timed(calls, len(calls)), alg)
        if rf.packed_supported(t, in_dim):
            # the same rf_matvec calls on GGUF bytes with the repack cache on:
            # the first call on each copy packs it, the timed ones hit
            ctx.matvec_cache(len(ws) * wbytes)
            for c in calls:
                c()
            ctx.synchronize()
            record(name, "matvec (GGUF, repack cache)", timed(calls, len(calls)), alg)
            ctx.matvec_cache(0)
            ps = []
            for i, w in enumerate(ws):
                p = ctx.empty((wbytes,), "uint8", charge=f"kbench:{name}:p{i}")
                rf.pack_weights(ctx, t, w, out_dim, in_dim, p)
                ps.append(p)
            calls = [lambda p=p: rf.matvec_packed(ctx, t, p, (out_dim, in_dim), x, y) for p in ps]
            record(name, "matvec_packed", timed(calls, len(calls)), alg)
            for p in ps:
                p.free()
        for a in ws + [x, y]:
            a.free()

    qh, kvh, hd = 32, 8, 128
    for L in (512, 2048, 8192):
        hist = L - 1
        kvb = hist * kvh * hd * 4
        copies = min(96, max(2, -(-(int(1.2 * 2 ** 30)) // (2 * kvb))))
        kv = []
        for i in range(copies):
            kh = ctx.array(rng.normal(0, 1, hist * kvh * hd).astype(np.float32), f"kbench:att{L}:k{i}")
            vh = ctx.array(rng.normal(0, 1, hist * kvh * hd).astype(np.float32), f"kbench:att{L}:v{i}")
            kv.append((kh, vh))
        q = ctx.array(rng.normal(0, 1, qh * hd).astype(np.float32), f"kbench:att{L}:q")
        kc = ctx.array(rng.normal(0, 1, kvh * hd).astype(np.float32), f"kbench:att{L}:kc")
        vc = ctx.array(rng.normal(0, 1, kvh * hd).astype(np.float32), f"kbench:att{L}:vc")
        o = ctx.empty((qh * hd,), charge=f"kbench:att{L}:o")

        def att(kh, vh):
            rf.apply_rope(ctx, q, kc, hist, hd, qh, kvh, 10000.0)
            rf.attention_checked(ctx, q, kh, vh, kc, vc, hist, qh, kvh, hd, out=o)

        calls = [lambda kh=kh, vh=vh: att(kh, vh) for kh, vh in kv]
        alg = 2 * L * kvh * hd * 4 + 2 * qh * hd * 4
        record(f"attention 32q/8kv hd128 L={L}", f"rope+attention ({copies} K/V copies)",
               timed(calls, len(calls)), alg)
        for kh, vh in kv:
            kh.free()
            vh.free()
        for a in (q, kc, vc, o):
            a.free()
    ctx.close()
    return out


def pinned_h2d_gbs(ctx, nbytes: int = 256 << 20, reps: int = 8) -> float:
    """Host-link peak for config 5's roofline: hipMemcpyAsync of a pinned
    (hipHostMalloc) buffer to device memory on the copy stream, HIP events."""
    import ctypes as C

    from ramforge_amd import _lib

    hp = C.c_void_p()
    _lib.check(ctx.lib.rf_pinned_alloc(ctx.handle, nbytes, C.byref(hp)))
    dev = ctx.empty((nbytes,), "uint8", charge="bench:h2d")
    try:
        C.memset(hp.value, 1, nbytes)
        st = ctx.copy_stream
        _lib.check(ctx.lib.rf_upload_async(ctx.handle, dev.ptr, hp.value, nbytes, st))  # warm
        e0, e1 = ctx.event(), ctx.event()
        ctx.record(e0, st)
        for _ in range(reps):
            _lib.check(ctx.lib.rf_upload_async(ctx.handle, dev.ptr, hp.value, nbytes, st))
        ctx.record(e1, st)
        ms = ctx.elapsed_ms(e0, e1)
        ctx.destroy_event(e0)
        ctx.destroy_event(e1)
    finally:
        dev.free()
        ctx.lib.rf_pinned_free(ctx.handle, hp.value)
    return nbytes * reps / (ms * 1e-3) / 1e9


def config5_bench(rf, syn, tokens: int, prompt_len: int, policy: int, persistent: int = 0,
                  model_file=None, units: int = 1) -> dict:
    """8B shape, Q4_K body + Q6_K output, VRAM budget 4 GiB:
    the layers that do not fit stream from pinned host memory each token
    (layer cache on the device with LRU or next-use eviction, uploads on the
    copy streams overlapped with the previous layers' kernels).  persistent:
    0 keeps the embedding and output resident by the reference's 25% rule,
    3 keeps the embedding table in mapped host memory (a step reads one
    row), leaving its VRAM to cached layers.  model_file: (path, spans) of
    the block tensors written by synthetic.write_model_file, read on every
    layer load through the library's pread reader instead of kept in pinned
    host memory; the model's worker thread reads the next layer to load into
    one of two pinned layer buffers while the pass runs (read-ahead, on by
    default for that reader).  units: streaming units per layer (2:
    attention tensors with the norms | gate, up, down; 3: attention | gate,
    up | down), so the budget also keeps part of a layer
    (rf_model_set_stream_units)."""
    import numpy as np

    cfg = syn.CONFIG_8B
    budget = 4 << 30
    specs = syn.llama_specs(cfg, syn.Q4_K, output_type=syn.Q6_K, seed=5)
    link = pinned_h2d_gbs(rf.Context(0))  # in a context of its own: the budgeted one is full
    log(f"config 5: pinned host-to-device copy peak {link:.1f} GB/s")
    ctx = rf.Context(0, budget)
    t0 = time.perf_counter()
    # context 8192 (2 GiB of f32 K/V at full length), the cache starting at the
    # prompt's length and growing in 256-position chunks as the reference's does
    if model_file is None:
        m = syn.build_device_model(ctx, cfg, specs, cfg["context_length"], stream_cache_bytes=budget,
                                   cache_policy=policy, kv_initial=prompt_len, persistent_policy=persistent)
    else:
        m = syn.build_file_model(ctx, cfg, specs, model_file[0], model_file[1], cfg["context_length"], budget,
                                 cache_policy=policy, kv_initial=prompt_len, persistent_policy=persistent)
    if units > 1:
        m.set_stream_units(units)
    fixed = ctx.vram_used
    layer = syn.weight_bytes([s for s in specs if s.name.startswith("blk.0.")])
    log(f"config 5: built in {time.perf_counter() - t0:.1f} s; fixed VRAM {fixed / 1e9:.2f} GB, "
        f"layer {layer / 1e6:.1f} MB, budget {budget / 2 ** 30:.0f} GiB")
    prompt = [int(t) for t in np.random.default_rng(5).integers(0, cfg["vocab_size"], prompt_len)]
    t0 = time.perf_counter()
    m.prefill(prompt)  # batched: each streamed layer is uploaded once per chunk (up to 512 tokens)
    prompt_s = time.perf_counter() - t0
    pre = m.residency_stats()
    log(f"config 5: prompt {prompt_len} tokens (batched prefill) in {prompt_s:.2f} s; {pre}")
    # the greedy loop of rf_model_generate (generate_impl): the KV cache grows
    # to at most the positions the request needs (prompt + tokens)
    t0 = time.perf_counter()
    gen = m.generate([], tokens)
    wall = time.perf_counter() - t0
    st = m.residency_stats()
    up = st["uploaded_bytes"] - pre["uploaded_bytes"]
    where = ("read from the model file on every layer load (pread, read ahead of the pass into two pinned "
             "layer buffers)" if model_file is not None else "streamed from pinned host memory")
    out = {"workload": "config 5: 8B shape, Q4_K body + Q6_K output, context 8192, 4 GiB VRAM budget, layers "
                       f"{where}, KV cache grown in 256-position chunks",
           "pinned_host_bytes": m.host_bytes(),
           "cache_policy": ["lru", "next-use"][policy],
           "stream_units_per_layer": units,
           "persistent": {0: "embedding and output resident (25% rule)",
                          3: "embedding in mapped host memory, output resident"}[persistent],
           "tokens": tokens, "tok_s": round(tokens / wall, 3),
           "kv_positions": m.kv_positions(),
           "ms_per_token": round(wall * 1e3 / tokens, 2), "uploaded_GB_per_token": round(up / tokens / 1e9, 3),
           "prompt_tokens": prompt_len, "prompt_prefill_s": round(prompt_s, 3),
           "host_to_device_GBs": round(up / wall / 1e9, 2), "pinned_h2d_peak_GBs": round(link, 2),
           "host_link_frac": round(up / wall / 1e9 / link, 4), "cache": st, "vram_peak_bytes": ctx.vram_peak,
           "vram_budget_bytes": budget, "fixed_vram_bytes": fixed, "layer_bytes": layer,
           "tokens_head": gen[:8]}
    log(f"config 5: {out['tok_s']} tok/s, {out['uploaded_GB_per_token']} GB/token uploaded at "
        f"{out['host_to_device_GBs']} GB/s")
    m.close()
    ctx.close()
    return out


def prefill_bench(ctx, m, cfg, rf, prompt, long_len: int) -> dict:
    """Prompt forwarding on the resident 8B-shape model: the reference's loop
    (one forward per token, inference.rs:580-592) against rf_model_prefill
    (chunks of up to 512 tokens, projections as packed-weight GEMMs on the matrix cores),
    and a long batched prompt.  Untimed warmup prefill first (workspace, LDS
    attributes)."""
    import numpy as np

    m.reset()
    t0 = time.perf_counter()
    for p, t in enumerate(prompt):
        m.forward(t, p)
    tbt = time.perf_counter() - t0
    m.reset()
    m.prefill(prompt[:8])
    m.reset()
    t0 = time.perf_counter()
    m.prefill(prompt)
    batched = time.perf_counter() - t0
    m.reset()
    lp = [int(t) for t in np.random.default_rng(12).integers(0, cfg["vocab_size"], long_len)]
    t0 = time.perf_counter()
    m.prefill(lp)
    long_s = time.perf_counter() - t0
    m.reset()
    d, f = cfg["embedding_length"], cfg["feed_forward_length"]
    qd = cfg["head_count"] * cfg["head_dim"]
    kvd = cfg["head_count_kv"] * cfg["head_dim"]
    params = cfg["block_count"] * (d * (qd + 2 * kvd) + qd * d + 2 * d * f + f * d)
    chunks = -(-long_len // 512)  # each reads the weights once
    useful = 2.0 * long_len * params / long_s / 1e12
    out = {"prompt_tokens": len(prompt), "token_by_token_ms": round(tbt * 1e3, 2),
           "batched_ms": round(batched * 1e3, 2), "speedup": round(tbt / batched, 1),
           "long_prompt_tokens": long_len, "long_batched_ms": round(long_s * 1e3, 2),
           "long_tok_s": round(long_len / long_s, 1),
           "long_useful_TFLOPs": round(useful, 2),
           "long_mfma_frac_bf16": round(3 * useful / PEAK_BF16_TFLOPS, 4),
           "long_weight_GBs": round(chunks * 1.0625 * params / long_s / 1e9, 1)}
    log(f"prefill: {len(prompt)} tokens token-by-token {tbt * 1e3:.1f} ms, batched {batched * 1e3:.1f} ms "
        f"({tbt / batched:.1f}x); {long_len} tokens batched {long_s * 1e3:.1f} ms = {long_len / long_s:.0f} tok/s, "
        f"{useful:.1f} useful TFLOP/s ({3 * useful / PEAK_BF16_TFLOPS:.1%} of bf16 MFMA peak with the 3-piece split)")
    return out


def config4_bench(rf, syn, tokens: int = 128, prompt_len: int = 32) -> dict:
    """random-init llama, 16 layers, d 2048, 32/8 heads, FFN
    8192, vocab 32000, Q8_0 everywhere, fully resident; 32-token prompt, 128
    greedy tokens.  Timed: the prompt token by token (the reference's loop) and
    batched (after an untimed batched pass that allocates the prefill
    workspace, as prefill_bench does), then the 128 greedy tokens as device
    decode steps (hipGraph replay; graphs captured in an untimed first pass)."""
    import numpy as np

    cfg = syn.CONFIG_4
    specs = syn.llama_specs(cfg, syn.Q8_0, seed=4)
    wbytes = syn.weight_bytes(specs)
    ctx = rf.Context(0)
    m = syn.build_device_model(ctx, cfg, specs, prompt_len + tokens + 8)
    prompt = [int(t) for t in np.random.default_rng(4).integers(0, cfg["vocab_size"], prompt_len)]
    t0 = time.perf_counter()
    for p, t in enumerate(prompt):
        m.forward(t, p)
    tbt = time.perf_counter() - t0
    m.use_graph(True)
    m.decode_steps(tokens)  # captures the regimes' graphs
    ctx.synchronize()
    m.reset()
    m.prefill(prompt)  # untimed: workspace and kernel attributes
    m.reset()
    t0 = time.perf_counter()
    m.prefill(prompt)
    batched = time.perf_counter() - t0
    t0 = time.perf_counter()
    m.decode_steps(tokens)
    ctx.synchronize()
    wall = time.perf_counter() - t0
    gen = m.read_tokens(tokens)
    # per launch group: HIP events around back-to-back eager launches at the
    # position the decode ended
    m.use_graph(False)
    groups = {}
    for kind in ("qkv", "attention", "oproj", "gateup", "down", "logits"):
        ms, b, _ = m.time_kernel(kind, 4)
        groups[kind] = {"us_per_launch": round(ms * 1e3, 2), "bytes_per_launch": b,
                        "kernel": m.kernel_name(kind) if kind != "attention" else ""}
    out = {"workload": "config 4: 16 layers, d 2048, 32/8 heads, FFN 8192, vocab 32000, Q8_0, resident",
           "prompt_tokens": prompt_len, "prompt_token_by_token_ms": round(tbt * 1e3, 2),
           "prompt_batched_ms": round(batched * 1e3, 2), "tokens": tokens, "tok_s": round(tokens / wall, 1),
           "ms_per_token": round(wall * 1e3 / tokens, 4), "weights_bytes_per_token": wbytes,
           "roofline_tok_s_at_peak": round(PEAK_HBM_GBS * 1e9 / wbytes, 1),
           "tokens_head": gen[:8], "per_group": groups}
    log(f"config 4: prompt {tbt * 1e3:.1f} ms token by token, {batched * 1e3:.1f} ms batched; "
        f"{out['tok_s']} tok/s decode ({out['ms_per_token']} ms/token; roofline {out['roofline_tok_s_at_peak']})")
    m.close()
    ctx.close()
    return out


def main() -> int:
    ap = argparse.ArgumentParser(description=__doc__.split("\n")[0])
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=128)
    ap.add_argument("--warmup", type=int, default=8)
    ap.add_argument("--prompt", type=int, default=32)
    ap.add_argument("--no-graph", action="store_true", help="eager launches instead of hipGraph replay")
    ap.add_argument("--cpu-steps", type=int, default=6, help="CPU baseline greedy steps (the first one is warmup)")
    ap.add_argument("--ctx-decode", default="2048,8192",
                    help="context lengths (comma separated) at which decode tok/s is also measured ('' to skip)")
    ap.add_argument("--ctx-steps", type=int, default=32)
    ap.add_argument("--skip-cpu", action="store_true")
    ap.add_argument("--prefill-tokens", type=int, default=512,
                    help="long batched prompt for the prefill measurement (0: skip the prefill measurement)")
    ap.add_argument("--prefill-only", action="store_true", help="only the prefill measurement (for rocprofv3)")
    ap.add_argument("--kernel-reps", type=int, default=4)
    ap.add_argument("--tile-bytes", type=int, default=0, help="matvec LDS tile bytes (tuning)")
    ap.add_argument("--kernels", action="store_true",
                    help="kernel-level BASELINE configs 1-3 (matvec formats/shapes, attention contexts) instead of "
                         "the decode benchmark; prints one JSON line")
    ap.add_argument("--config4", action="store_true",
                    help="BASELINE config 4 (16-layer d2048 Q8_0 model): prompt and 128-token decode timings")
    ap.add_argument("--config5", type=int, default=0, metavar="TOKENS",
                    help="BASELINE config 5 (Q4_K/Q6_K 8B under a 4 GiB VRAM budget, layer streaming) with TOKENS "
                         "greedy tokens; prints one JSON line")
    ap.add_argument("--attention-probe", type=int, default=0, metavar="L",
                    help="only launch RoPE + attention at context L on 4 K/V copies and a 256 MiB device copy, for "
                         "rocprofv3 --pmc runs")
    ap.add_argument("--matvec-probe", default="", metavar="TYPE,OUT,IN",
                    help="only launch the GGUF-layout and packed matvec of one shape on 4 weight copies and a 256 "
                         "MiB device copy, for rocprofv3 --pmc runs")
    ap.add_argument("--traffic-probe", action="store_true",
                    help="only launch the dominant kernel (32 gate/up launches) and a 256 MiB device copy, "
                         "for rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE runs")
    args = ap.parse_args()
    world = int(os.environ.get("WORLD_SIZE", "1"))
    if args.gpus != 1 or world != 1:
        print("bench.py measures the decode hot path on ONE GPU only: this build has no multi-GPU path "
              "(no collectives or sharding); run with --gpus 1.", file=sys.stderr)
        return 2
    model_graph = not (args.kernels or args.attention_probe or args.matvec_probe or args.traffic_probe
                       or args.prefill_only or args.config5)
    if model_graph and not args.no_graph and under_tracer():
        # Three kernel traces of the graph-replayed decode step crashed on the
        # host inside rf_model_decode_steps (a profiler callback under the HIP
        # runtime reading an unmapped address), cause not established.
        print("bench.py: graph-replayed decode is not run under rocprofv3 (the kernel tracer has crashed inside "
              "the decode step's capture/replay); trace the same kernels with --no-graph.", file=sys.stderr)
        return 2

    import numpy as np

    import ramforge_amd as rf
    from ramforge_amd import synthetic as syn

    if args.tile_bytes:
        rf.tune_matvec_tile_bytes(args.tile_bytes)
    if args.config4:
        print(json.dumps({"config4": config4_bench(rf, syn)}), flush=True)
        return 0
    if args.attention_probe:
        return attention_probe(rf, args.attention_probe)
    if args.matvec_probe:
        return matvec_probe(rf, args.matvec_probe)
    if args.config5:
        res = [config5_bench(rf, syn, args.config5, args.prompt, policy, persistent, units=k)
               for policy, persistent, k in ((1, 3, 2), (1, 3, 1), (1, 0, 1), (0, 0, 1))]
        # the same model with its block tensors read from a model file
        import shutil
        import tempfile

        specs5 = syn.llama_specs(syn.CONFIG_8B, syn.Q4_K, output_type=syn.Q6_K, seed=5)
        d = tempfile.mkdtemp(prefix="rf_config5_")
        try:
            need = syn.weight_bytes([s_ for s_ in specs5 if s_.name.startswith("blk.")])
            if shutil.disk_usage(d).free > need + (2 << 30):
                path = os.path.join(d, "config5_blocks.bin")
                t0 = time.perf_counter()
                with rf.Context(0) as wctx:
                    spans = syn.write_model_file(wctx, specs5, path)
                log(f"config 5: wrote {need / 1e9:.2f} GB of block tensors to {path} in "
                    f"{time.perf_counter() - t0:.1f} s")
                for k in (2, 1):
                    res.append(config5_bench(rf, syn, args.config5, args.prompt, 1, 3, model_file=(path, spans),
                                             units=k))
            else:
                log("config 5: not enough free disk for the model file; file-read row skipped")
        finally:
            shutil.rmtree(d, ignore_errors=True)
        print(json.dumps({"config5": res}), flush=True)
        return 0
    if args.kernels:
        rows = kernel_bench(rf, syn, use_graph=not args.no_graph)
        print(json.dumps({"kernels": rows, "peak_GBs": PEAK_HBM_GBS, "timing": "hipGraph replay" if not args.no_graph
                          else "eager launches (host-bound; see the rocprof trace)"}), flush=True)
        return 0
    cfg = syn.CONFIG_8B
    specs = syn.llama_specs(cfg, syn.Q8_0, seed=8)
    wbytes = syn.weight_bytes(specs)
    embd = syn.weight_bytes([s_ for s_ in specs if s_.name == "token_embd.weight"])
    # a step reads one row of the embedding table, every other weight once
    step_wbytes = wbytes - embd + embd // cfg["vocab_size"]
    ctx_lens = [int(v) for v in args.ctx_decode.split(",") if v.strip()]
    cap = max([args.prompt + args.warmup + args.steps, args.prefill_tokens] + ctx_lens) + 8
    cap = min(cap, cfg["context_length"])
    ctx = rf.Context(0)
    name, cus = ctx.device_info()
    log(f"device {name}, {cus} CUs; building 8B-shape Q8_0 model ({wbytes / 1e9:.2f} GB) in HBM")
    m = syn.build_device_model(ctx, cfg, specs, cap)
    if args.traffic_probe:
        return traffic_probe(ctx, m, cfg, rf)
    prompt = [int(t) for t in np.random.default_rng(8).integers(0, cfg["vocab_size"], args.prompt)]
    pre = None
    if args.prefill_tokens:
        pre = prefill_bench(ctx, m, cfg, rf, prompt, args.prefill_tokens)
        if args.prefill_only:
            print(json.dumps({"prefill": pre}), flush=True)
            return 0
    t0 = time.perf_counter()
    m.prefill(prompt)
    log(f"prompt of {args.prompt} tokens forwarded (batched) in {time.perf_counter() - t0:.3f} s")
    m.use_graph(not args.no_graph)
    m.decode_steps(args.warmup)
    ctx.synchronize()

    t0 = time.perf_counter()
    m.decode_steps(args.steps)
    ctx.synchronize()
    wall = time.perf_counter() - t0
    toks = m.read_tokens(args.steps)
    tok_s = args.steps / wall
    ms_step = wall * 1e3 / args.steps
    log(f"decode: {args.steps} steps in {wall * 1e3:.1f} ms -> {tok_s:.1f} tok/s ({ms_step:.3f} ms/step)")

    # live per-group kernel times (HIP events on the compute stream)
    m.use_graph(False)
    per_token_bytes = 0
    breakdown = {}
    for kind in ("qkv", "attention", "oproj", "gateup", "down", "logits"):
        ms, b, n = m.time_kernel(kind, args.kernel_reps)
        per_tok = 1 if kind == "logits" else cfg["block_count"]
        breakdown[kind] = {"us_per_launch": round(ms * 1e3, 3), "launches_per_token": per_tok,
                           "bytes_per_launch": b, "GBs": round(b / (ms * 1e-3) / 1e9, 1)}
        per_token_bytes += b * per_tok
    kernel_ms = sum(v["us_per_launch"] * v["launches_per_token"] for v in breakdown.values()) / 1e3
    dom = max(breakdown, key=lambda k: breakdown[k]["us_per_launch"] * breakdown[k]["launches_per_token"])
    d = breakdown[dom]
    achieved = d["bytes_per_launch"] / (d["us_per_launch"] * 1e-6) / 1e9
    traffic = None
    kname = dominant_kernel(m) if dom == "gateup" else dom
    tpath = os.path.join(ROOT, "profiles", "gateup_q8_0_8b_traffic.json")
    if dom == "gateup" and os.path.exists(tpath):
        try:
            tj = json.load(open(tpath))
            # only a measurement of the exact kernel instance that ran counts
            traffic = tj.get("bytes_per_launch") if tj.get("kernel") == kname else None
        except (OSError, ValueError):
            traffic = None
    # the same figure from the committed rocprofv3 trace of this kernel
    t_us = trace_mean_us(kname)
    roofline = {"bound": "hbm", "achieved": round(achieved, 1), "peak": PEAK_HBM_GBS, "unit": "GB/s",
                "frac": round(achieved / PEAK_HBM_GBS, 4), "traffic": traffic, "kernel": kname,
                "timing": "HIP events around back-to-back launches on the compute stream",
                "trace_us_per_launch": t_us,
                "frac_from_trace": None if t_us is None else round(d["bytes_per_launch"] / (t_us * 1e-6) / 1e9
                                                                    / PEAK_HBM_GBS, 4)}
    log(f"dominant group {dom}: {d['us_per_launch']} us/launch, {achieved:.0f} GB/s "
        f"({achieved / PEAK_HBM_GBS:.1%} of peak); kernel time per token {kernel_ms:.3f} ms")
    ctx_decode = {}
    for n in ctx_lens:
        ctx_decode[str(n)] = context_decode(ctx, m, cfg, min(n, cap - args.ctx_steps - 4), args.ctx_steps,
                                            not args.no_graph)
    # the GPU's greedy tokens from the start the CPU baseline uses
    m.use_graph(False)
    m.reset()
    m.forward(prompt[0], 0)
    m.decode_steps(max(args.cpu_steps, 1))
    gpu_cpu_start = m.read_tokens(max(args.cpu_steps, 1))
    mv = matvec_q8_0_gbs(ctx, rf, syn)
    log(f"Q8_0 4096x4096 matvec: {mv['achieved_GBs']} GB/s")
    m.close()
    ctx.close()

    cpu = None
    cross = None
    if not args.skip_cpu:
        log(f"CPU baseline: {args.cpu_steps} greedy steps of the oracle restatement (first one warmup)")
        cpu, cpu_toks = cpu_baseline(cfg, specs, prompt[0], args.cpu_steps)
        cross = {"start": "prompt token 0 at position 0", "cpu_tokens": cpu_toks,
                 "gpu_tokens": gpu_cpu_start[:len(cpu_toks)], "match": cpu_toks == gpu_cpu_start[:len(cpu_toks)]}
        log(f"CPU and GPU greedy tokens from the same start {'match' if cross['match'] else 'DIFFER'}: "
            f"{cpu_toks} vs {cross['gpu_tokens']}")

    line = {
        "metric": METRIC, "value": round(tok_s, 2), "unit": "tok/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(ms_step, 4), "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": "f32", "data": "synthetic",
        "config": {"workload": "greedy decode, 1 token per step, llama 8B shape, Q8_0 weights resident in HBM",
                   "layers": cfg["block_count"], "d_model": cfg["embedding_length"],
                   "heads": [cfg["head_count"], cfg["head_count_kv"]], "ffn": cfg["feed_forward_length"],
                   "vocab": cfg["vocab_size"], "prompt_tokens": args.prompt,
                   "weights_bytes_per_token": step_wbytes, "model_weight_bytes": wbytes,
                   "hip_graph": not args.no_graph},
        "roofline": roofline,
        "cpu_baseline": cpu,
        "cpu_gpu_tokens": cross,
        "decode_at_context": ctx_decode,
        "roofline_tok_s_at_peak": round(PEAK_HBM_GBS * 1e9 / per_token_bytes, 1),
        "kernel_ms_per_token": round(kernel_ms, 4),
        "breakdown": breakdown,
        "matvec_q8_0_4096x4096": mv,
        "prefill": pre,
        "tokens_head": toks[:8],
        "device": name,
    }
    print(json.dumps(line), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
