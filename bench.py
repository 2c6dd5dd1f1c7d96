#!/usr/bin/env python3
"""Benchmark of the INT8 KV-cache path on one MI355X.

Metric: "30K-prefill INT8-KV attn ms/layer (MFMA %); 128K decode KV-read GB/s".

* step (``value``, ms per layer): config 3 — a 30720-token causal prompt of one
  full-attention layer in 60 chunks of 512 tokens. Per chunk, the engine's INT8 sequence
  with fused preparation, the one the reference measured at 30K (Prefill.cs:249-251,261):
  attention_prepare_fused_int8 (norm, RoPE, grouped FP16 Q, gate, INT8 append) ->
  attention_online_int8 on the prepared query (+ split combine). Inputs (FP32 qkv, K, V)
  are resident in HBM before timing; synthetic N(0,1) with K channels {30,31,62,63} x 20;
  16 Q / 2 KV heads, d = 256.
* decode (extra keys): config 4 — cache grown from 4096 tokens by doubling with device
  copies while being filled to 131072 tokens, pre-grown to 262144, then 256 sequential
  single-token steps over L = 131073..131328, each one attention_decode_append_int8 dispatch
  per layer (batch_rope_int8 with M = 1 and the attention, fused; + split combine).
* roofline: prefill attention kernel against the dense FP16 MFMA peak (2.5 PFLOP/s),
  decode kernel against HBM (8 TB/s); kernel durations from HIP events on the library's
  stream over the timed region.
* cpu_baseline: the C oracle (FP64, the reference's checker arithmetic) on the host threads,
  median of 5 runs each of config 1, config 2, one 131072-token decode step, and config 3's
  last 512-query chunk extrapolated by the causal flop ratio (``value``).
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(ROOT, "llm-bootstrap-qwen3.6-35b-dotnet-metal_amd"))

from bootstrap_hip import Device, KernelArgs, engine  # noqa: E402

METRIC = "30K-prefill INT8-KV attn ms/layer (MFMA %); 128K decode KV-read GB/s"
MFMA_PEAK_TFLOPS = 2500.0      # MI355X dense FP16/BF16
HBM_PEAK_GBS = 8000.0          # MI355X HBM3E
OUTLIER_CHANNELS = [30, 31, 62, 63]


def log(msg: str) -> None:
    print(msg, file=sys.stderr, flush=True)


def synthetic(rng, shape, outliers=False):
    x = rng.standard_normal(shape, dtype=np.float32)
    if outliers:
        x[..., OUTLIER_CHANNELS] *= 20
    return x


def upload(device, array):
    b = device.allocate(array.nbytes)
    b.write(array)
    return b


# the INT8 prefill attention kernels: the main one (its FP16-KV control: prefill_w64_fp16_kernel) and
# the multi-row kernel that serves the chunks over the first keys
PREFILL_INT8_KERNELS = ["prefill_w64_kernel", "rows_int8_half_query_kernel"]


def kernel_stats(device, names):
    stats = {k["kernel"]: k for k in device.read_wall_timing()["kernels"]}
    out = {}
    for name in names:
        if name in stats:
            out[name] = (stats[name]["gpu_ms"], int(stats[name]["count"]))
    return out


def measured_traffic(kernel: str):
    """HBM bytes per launch of ``kernel`` (read + write) from the committed rocprofv3 PMC
    summary (FETCH_SIZE / WRITE_SIZE, scaled by a plain device copy of known size), or None."""
    path = os.path.join(ROOT, "profiles", "traffic.json")
    try:
        with open(path) as f:
            entry = json.load(f)["kernels"][kernel]
    except (OSError, KeyError, ValueError):
        return None
    return int(round((entry["fetch_mb"] + entry["write_mb"]) * 1e6))


def measured_counters(kernel: str):
    """Counter-derived utilisation of ``kernel`` from the committed rocprofv3 PMC summary
    (profiles/counters.json: MFMA busy, LDS active, bank conflicts), or None."""
    path = os.path.join(ROOT, "profiles", "counters.json")
    try:
        with open(path) as f:
            entry = json.load(f)["kernels"][kernel]
    except (OSError, KeyError, ValueError):
        return None
    return {k: entry[k] for k in ("mfma_busy", "lds_active", "lds_bank_conflicts_per_access")}


def prefill_flops(pos: int, rows: int) -> float:
    # 4 * d * H * sum over rows of visible keys (QK and PV, 2 flop per MAC)
    return 4.0 * 256 * 16 * (rows * pos + rows * (rows + 1) / 2)


# --------------------------------------------------------------------------- prefill

class PrefillWorkload:
    """Config 3 per chunk as the reference's measured 30K INT8 run issues it (fused preparation,
    Prefill.cs:249-251,261; 160 attention calls among 340 attention-and-preparation dispatches,
    docs/INT8_30K_NEXT_PROFILE_20261104.md:36-45): attention_prepare_fused_int8 (Q/K RMS norm,
    RoPE, grouped FP16 Q, gate split, INT8 append) -> attention_online_int8_q32_k256_r2 on the
    prepared query (+ split combine). Synthetic qkv [tokens][16][q|gate][256], K with outlier
    channels, V, all ~N(0,1); norm weights 0 (RMS normalisation with w + 1 = 1)."""

    def __init__(self, device, tokens=30720, chunk=512, seed=0):
        self.device, self.tokens, self.chunk = device, tokens, chunk
        rng = np.random.default_rng(seed)
        log(f"prefill: generating {tokens} tokens of synthetic qkv/K/V")
        self.qkv = upload(device, synthetic(rng, (tokens, 8192)))
        self.k = upload(device, synthetic(rng, (tokens, 2, 256), outliers=True))
        self.v = upload(device, synthetic(rng, (tokens, 2, 256)))
        self.q_norm = upload(device, np.zeros(256, np.uint16))
        self.k_norm = upload(device, np.zeros(256, np.uint16))
        self.gate = device.allocate(chunk * 16384)          # the chunk's gate, split out by the preparation
        self.out = device.allocate(chunk * 16384)           # the chunk's attention output
        self.cache = engine.Int8KvCache(device, context_window=engine.NATIVE_WINDOW, layers=1)
        self.cache.ensure_capacity(tokens)
        self.layer = self.cache.layers[0]
        self.workspace = engine.DeviceAttentionWorkspace(device)
        self.workspace.prepare(chunk)

    def step(self):
        d, layer, ws = self.device, self.layer, self.workspace
        d.begin()
        for pos in range(0, self.tokens, self.chunk):
            rows = min(self.chunk, self.tokens - pos)
            engine.prepare_fused(d, layer, self.qkv.at(pos * 32768), self.k.at(pos * 2048), self.v.at(pos * 2048),
                                 self.q_norm, self.k_norm, ws.packed_query, self.gate, rows, pos)
            ws.encode_int8(None, layer.key, layer.value, layer.key_scale, layer.value_scale, self.gate, self.out,
                           rows, pos, prepared_query=True)
        d.end()

    def flops(self):
        return sum(prefill_flops(pos, min(self.chunk, self.tokens - pos)) for pos in range(0, self.tokens, self.chunk))


# (history, query rows, the reference's GPU median in ms on an M5 Pro) of its INT8 online kernel
# (docs/INT8_30K_PREFILL_20261104.md:59-61)
REFERENCE_SHAPES = [(0, 33, 0.02408), (8192, 2048, 14.82842), (27900, 2048, 44.22633)]


def reference_shapes(work: PrefillWorkload, runs: int = 20):
    """attention_online_int8_q32_k256_r2 at the shapes the reference times it at, over config 3's
    cache: the query and gate prepared by attention_prepare_fused_int8 at those rows (which rewrites
    the same cache rows with the same bytes), then `runs` launches timed kernel-exact (attention
    kernel + split combine, averaged). The M5 Pro medians are context, not a same-node comparison."""
    d = work.device
    ws = engine.DeviceAttentionWorkspace(d)
    ws.prepare(2048)
    gate, out = d.allocate(2048 * 16384), d.allocate(2048 * 16384)
    layer = work.layer
    entries = []
    for history, rows, m5 in REFERENCE_SHAPES:
        d.begin()
        engine.prepare_fused(d, layer, work.qkv.at(history * 32768), work.k.at(history * 2048), work.v.at(history * 2048),
                             work.q_norm, work.k_norm, ws.packed_query, gate, rows, history)
        for _ in range(3):
            ws.encode_int8(None, layer.key, layer.value, layer.key_scale, layer.value_scale, gate, out, rows, history,
                           prepared_query=True)
        d.end()
        d.reset_wall_timing(kernels_exact=True)
        d.begin()
        for _ in range(runs):
            ws.encode_int8(None, layer.key, layer.value, layer.key_scale, layer.value_scale, gate, out, rows, history,
                           prepared_query=True)
        d.end()
        # small chunks run on the decode kernel or the multi-row kernel (their grouped FP16 query
        # variants) and, when split, their combine
        served = PREFILL_INT8_KERNELS + ["decode_int8_half_query_kernel"]
        ks = kernel_stats(d, served + ["prefill_combine_kernel", "decode_combine_kernel"])
        kernel = next(n for n in served if n in ks)
        attn = ks[kernel][0] / runs
        comb = sum(ks.get(n, (0.0, 0))[0] for n in ("prefill_combine_kernel", "decode_combine_kernel")) / runs
        flops = prefill_flops(history, rows)
        entries.append({"history": history, "rows": rows, "kernel": kernel, "attention_kernel_ms": round(attn, 5),
                        "combine_ms": round(comb, 5), "ms": round(attn + comb, 5),
                        "mfma_frac_attention_kernel": round(flops / (attn * 1e-3) / 1e12 / MFMA_PEAK_TFLOPS, 4),
                        "reference_m5pro_gpu_median_ms": m5})
    for b in (gate, out):
        b.dispose()
    ws.dispose()
    return {"what": "attention_online_int8_q32_k256_r2 at the reference's timed shapes (history, query rows), "
                    f"kernel-exact (the kernel that served the shape and its split combine), mean of {runs} launches "
                    f"over config 3's cache; the reference's figures are GPU "
                    "medians on an Apple M5 Pro (docs/INT8_30K_PREFILL_20261104.md:59-61), context only",
            "shapes": entries}


class Fp16ControlWorkload:
    """The same prompt with FP16 KV storage (config 3's side-by-side comparator), in the same
    shape: attention_prepare_fused (FP16 K/V) -> attention_online_q32_k256_s8_g8_r2 on the
    prepared query (+ split combine)."""

    def __init__(self, work: PrefillWorkload):
        self.work = work
        self.layer = engine.Fp16KvLayer(work.device, work.tokens)

    def step(self):
        w, d = self.work, self.work.device
        d.begin()
        for pos in range(0, w.tokens, w.chunk):
            rows = min(w.chunk, w.tokens - pos)
            engine.prepare_fused_fp16(d, self.layer, w.qkv.at(pos * 32768), w.k.at(pos * 2048), w.v.at(pos * 2048),
                                      w.q_norm, w.k_norm, w.workspace.packed_query, w.gate, rows, pos)
            engine.encode_online_fp16(w.workspace, None, self.layer, w.gate, w.out, rows, pos, prepared_query=True)
        d.end()


def host_threads():
    """(threads, nproc, affinity) for the CPU baseline: the CPU share the job is granted
    (OMP_NUM_THREADS where the scheduler sets it, as on the GPU boxes), else every CPU this
    process may run on."""
    affinity = len(os.sched_getaffinity(0))
    env = os.environ.get("OMP_NUM_THREADS", "")
    threads = min(int(env), affinity) if env.isdigit() and int(env) > 0 else affinity
    return threads, os.cpu_count(), affinity


def _spread(times_s):
    t = sorted(x * 1000.0 for x in times_s)
    return {"median_ms": round(float(np.median(t)), 3), "min_ms": round(t[0], 3), "max_ms": round(t[-1], 3),
            "runs": len(t)}


def _timed(fn, runs):
    times = []
    for _ in range(runs):
        t0 = time.perf_counter()
        fn()
        times.append(time.perf_counter() - t0)
    return times


def _rotated_queries(q_host, pos):
    """Partial RoPE of FP32 queries [rows][16][256] at positions pos.. (Int8KvTests.cs:13-18),
    vectorised in FP64; input preparation, not timed."""
    q = q_host.astype(np.float64)
    angle = (pos + np.arange(q.shape[0]))[:, None] * 10_000_000.0 ** (-2.0 * np.arange(32) / 64)
    c, s = np.cos(angle)[:, None, :], np.sin(angle)[:, None, :]
    a, b = q[:, :, :32].copy(), q[:, :, 32:64].copy()
    q[:, :, :32], q[:, :, 32:64] = a * c - b * s, b * c + a * s
    return np.ascontiguousarray(q.astype(np.float32).ravel())


def cpu_baseline(work: "PrefillWorkload", dec: "DecodeWorkload", y_last, runs: int = 5):
    """The reference's scalar CPU checker restated in C (the oracle: FP64 attention of
    Int8KvTests.cs:130-158 over the INT8 cache, append of Int8KvTests.cs:116-118), work split over
    (row, head) for attention and over tokens for append, on the host threads; median of `runs`
    runs of each workload on the same seeded inputs as the GPU path. ``value`` is config 3 in
    ms/layer: its last 512-query chunk timed in full and scaled by the causal flop ratio to the
    whole 30720-token layer (labelled as extrapolated). Also the parity check of what was timed:
    ``y_last`` (the INT8 path's output of the last chunk) against the same FP64 attention, with the
    bar rel-L2 <= 1e-3, max-abs <= 2e-3 and the per-element bound of Int8KvTests.cs:154-156, and
    the finished cache's V codes and scales against the oracle's quantizer."""
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    from oracle_lib import Oracle
    threads, nproc, affinity = host_threads()
    oracle = Oracle()
    oracle.threads = threads
    entries = {}

    # config 1: append 512 tokens of N(0,1) K/V (seed 0/1), one FP32 decode query over all 512
    k1 = oracle.normal(512 * 512, 0).reshape(512, 2, 256)
    v1 = oracle.normal(512 * 512, 1).reshape(512, 2, 256)
    q1, g1 = oracle.normal(4096, 2), np.zeros(4096, np.float32)
    c1 = oracle.empty_cache(512)

    def config1():
        oracle.store_mt(k1, v1, 0, *c1)
        oracle.attention(q1, *c1, g1, 1, 511, round_q_half=0)
    entries["config1_append512_decode"] = dict(_spread(_timed(config1, runs)), what="append 512 tokens + 1 decode query over 512 keys")

    # config 2: 4096-token causal prompt, 8 chunks of 512 (append + FP16-Q prefill per chunk)
    k2 = oracle.normal(4096 * 512, 20).reshape(4096, 2, 256)
    k2[:, :, OUTLIER_CHANNELS] *= 20
    v2 = oracle.normal(4096 * 512, 21).reshape(4096, 2, 256)
    q2, g2 = oracle.normal(4096 * 4096, 22), np.zeros(512 * 4096, np.float32)
    c2 = oracle.empty_cache(4096)

    def config2():
        for pos in range(0, 4096, 512):
            oracle.store_mt(k2[pos:pos + 512], v2[pos:pos + 512], pos, *c2)
            oracle.attention(q2[pos * 4096:(pos + 512) * 4096], *c2, g2, 512, pos, round_q_half=1)
    entries["config2_prefill4096"] = dict(_spread(_timed(config2, runs)), what="4096-token causal prefill in 8 chunks of 512 (append + attention)")

    # config 4: one decode step at 131072 context over the GPU-built layer (append 1 token +
    # attention over 131073 keys)
    if dec is not None:
        L = dec.context + 1
        layer = dec.cache.layers[0]
        cache4 = (layer.key.read(np.int8, L * 512), layer.value.read(np.int8, engine.int8_value_capacity(L) * 512),
                  layer.key_scale.read(np.float32, L * 2), layer.value_scale.read(np.float32, L * 2))
        k4 = dec.k_new.read(np.float32, 512).reshape(1, 2, 256)
        v4 = dec.v_new.read(np.float32, 512).reshape(1, 2, 256)
        q4 = _rotated_queries(dec.q.read(np.float32, 4096).reshape(1, 16, 256), dec.context)
        g4 = dec.gate.read(np.float32, 4096)

        def decode_step():
            oracle.store_mt(k4, v4, dec.context, *cache4)
            oracle.attention(q4, *cache4, g4, 1, dec.context, round_q_half=0)
        spread = _spread(_timed(decode_step, runs))
        spread["kv_read_gbs"] = round(1040 * L / (spread["median_ms"] * 1e-3) / 1e9, 2)
        entries["config4_decode_step_131072"] = dict(spread, what="append 1 token + decode over 131073 keys (one layer)")

    # config 3: the last 512-query chunk over the GPU-built 30720-token cache, extrapolated
    tokens, chunk = work.tokens, work.chunk
    pos = tokens - chunk
    layer = work.layer
    cache3 = (layer.key.read(np.int8, tokens * 512), layer.value.read(np.int8, engine.int8_value_capacity(tokens) * 512),
              layer.key_scale.read(np.float32, tokens * 2), layer.value_scale.read(np.float32, tokens * 2))
    # the last chunk's prepared query (grouped FP16 [2][rows][8][256], as the GPU attended it) and gate
    packed = work.workspace.packed_query.read(np.float16, chunk * 4096).reshape(2, chunk, 8, 256)
    q3 = np.ascontiguousarray(packed.transpose(1, 0, 2, 3).astype(np.float32).ravel())
    g3 = work.gate.read(np.float32, chunk * 4096)
    last = _spread(_timed(lambda: oracle.attention(q3, *cache3, g3, chunk, pos, round_q_half=1), runs))
    ratio = work.flops() / prefill_flops(pos, chunk)
    # parity of the timed chain (outside every timed region): the last chunk's output and the V cache
    ref, bound = oracle.attention(q3, *cache3, g3, chunk, pos, round_q_half=1, with_bound=True)
    err = np.abs(y_last.astype(np.float64) - ref)
    rel = float(np.linalg.norm(y_last.astype(np.float64) - ref) / np.linalg.norm(ref))
    v_host = work.v.read(np.float32, tokens * 512).reshape(tokens, 2, 256)
    okc, ovc, oks, ovs = oracle.empty_cache(tokens)
    oracle.store_mt(np.zeros_like(v_host), v_host, 0, okc, ovc, oks, ovs)
    v_equal = cache3[1].tobytes() == ovc.tobytes() and cache3[3].tobytes() == ovs.tobytes()
    parity = {"what": f"INT8 output of the last timed chunk (queries {pos}-{tokens - 1}) vs FP64 attention over the "
                      "device's cache and prepared FP16 query; V codes/scales of the 30720-token cache vs the oracle",
              "rel_l2": float(f"{rel:.4g}"), "max_abs": float(f"{err.max():.4g}"),
              "within_element_bound": bool(np.all(err <= bound / 256 + 1e-4)),
              "v_cache_bitwise": bool(v_equal),
              "pass": bool(rel <= 1e-3 and err.max() <= 2e-3 and np.all(err <= bound / 256 + 1e-4) and v_equal)}
    last["extrapolated_ms_per_layer"] = round(last["median_ms"] * ratio, 1)
    entries["config3_last_chunk"] = dict(last, what=f"queries {pos}-{tokens - 1} over {tokens} keys; x{ratio:.2f} causal flop ratio to the layer")
    return {"value": last["extrapolated_ms_per_layer"], "unit": "ms/layer", "cores": threads, "kind": "port",
            "nproc": nproc, "affinity_cpus": affinity,
            "sample": f"C restatement of the reference's FP64 CPU checker (Int8KvTests.cs:116-118,130-158) on {threads} "
                      f"host threads (nproc {nproc}), median of {runs} runs per workload; value = config 3's last "
                      f"512-query chunk ({last['median_ms'] / 1000:.2f} s) extrapolated x{ratio:.1f} by the causal flop "
                      f"ratio to the 30720-token layer",
            "entries": entries}, parity


# --------------------------------------------------------------------------- verify reader

def verify_block(dec, rows: int = 8, runs: int = 5):
    """The attention of a speculative verify block as the engine dispatches it (attention_verify_int8,
    Prefill.cs:269-285) for `rows` draft rows at the end of config 4's cache (layer 0), kernel-exact,
    mean of `runs` blocks."""
    d = dec.device
    layer = dec.cache.layers[0]
    length = dec.pos0 + dec.steps
    history = length - rows
    out = d.allocate(rows * 16384)
    p = KernelArgs(M=rows, K=length, Position=history)

    def block():   # (not in place, as the engine has it: the query serves every run)
        d.dispatch("attention_verify_int8", p, rows * 4096, 256, dec.q, layer.key, layer.value, dec.gate, out,
                   layer.key_scale, layer.value_scale)

    d.begin()
    block()
    d.end()
    d.reset_wall_timing(kernels_exact=True)
    d.begin()
    for _ in range(runs):
        block()
    d.end()
    ks = kernel_stats(d, ["rows_int8_kernel", "decode_combine_kernel"])
    us = {n: round(ms / runs * 1000, 2) for n, (ms, _) in ks.items()}
    out.dispose()
    return {"history": history, "rows": rows, "kernel_us": us, "total_us": round(sum(us.values()), 2),
            "kv_bytes": 1040 * length, "what": "one dispatch, four rows per work-group, and the splits' combine, "
                                               "kernel-exact, one layer"}


def verify_reader(dec, rows: int = 8, runs: int = 5):
    """The scalar reader (kernels.metal:147-166: batch_attention_scores_int8, attention_softmax,
    batch_attention_values_int8), which serves direct callers and verify blocks of more than 64 rows,
    for `rows` rows at the end of config 4's cache (layer 0), kernel-exact, mean of `runs` blocks."""
    d = dec.device
    layer = dec.cache.layers[0]
    length = dec.pos0 + dec.steps
    history = length - rows
    scores = d.allocate(rows * 16 * length * 4)
    out = d.allocate(rows * 16384)
    p = KernelArgs(M=rows, K=length, Position=history)

    def block():
        d.dispatch2d("batch_attention_scores_int8", p, length * 32, rows * 16, 128, dec.q, layer.key, scores,
                     layer.key_scale)
        d.dispatch("attention_softmax", KernelArgs(M=rows, K=length, Position=length - 1), rows * 16 * 256, 256, scores)
        d.dispatch("batch_attention_values_int8", p, rows * 4096, 128, scores, layer.value, dec.gate, out,
                   layer.value_scale)

    d.begin()
    block()
    d.end()
    d.reset_wall_timing(kernels_exact=True)
    d.begin()
    for _ in range(runs):
        block()
    d.end()
    names = ["scores_int8_kernel", "softmax_stats_kernel", "softmax_apply_kernel", "values_partial_kernel",
             "values_combine_kernel"]
    ks = kernel_stats(d, names)
    us = {n: round(ks[n][0] / runs * 1000, 2) for n in names if n in ks}
    for b in (scores, out):
        b.dispose()
    return {"history": history, "rows": rows, "kernel_us": us, "total_us": round(sum(us.values()), 2),
            "kv_bytes": 1040 * length,
            "what": "scores (INT8 MFMA, three-part query), softmax (chunk statistics, then normalize), values "
                    "(split-K FP16 MFMA, then the splits' sum with the gate), kernel-exact, one layer"}


# --------------------------------------------------------------------------- decode

class DecodeWorkload:
    """Config 4: single-token decode at 131072 context over the model's 10 full-attention
    layers (QwenEngine.cs:161-165 per layer): each step appends one token to every layer and
    attends over it. Ten layers of 136 MB do not fit the 256 MB last-level cache, so every
    layer's K/V comes from HBM as it does in the model (re-reading a single layer would be
    served partly from that cache)."""

    def __init__(self, device, context=131072, steps=256, layers=10, seed=1, fill_chunk=8192):
        self.device, self.context, self.steps = device, context, steps
        rng = np.random.default_rng(seed)
        self.cache = engine.Int8KvCache(device, context_window=engine.NATIVE_WINDOW, layers=layers)
        log(f"decode: filling {layers} layers x {context} tokens (capacity grows by doubling from {self.cache.capacity})")
        k_all = synthetic(rng, (context + steps, 2, 256), outliers=True)
        v_all = synthetic(rng, (context + steps, 2, 256))
        kb, vb = upload(device, k_all[:fill_chunk]), upload(device, v_all[:fill_chunk])
        for pos in range(0, context, fill_chunk):
            self.cache.ensure_capacity(pos + fill_chunk)       # PrefillBlock -> EnsureCacheCapacity
            kb.write(k_all[pos:pos + fill_chunk])
            vb.write(v_all[pos:pos + fill_chunk])
            device.begin()
            for layer in self.cache.layers:                    # the same rows in every layer
                engine.store_rows(device, layer, kb, vb, fill_chunk, pos)
            device.end()
        self.cache.ensure_capacity(context + steps)            # pre-grow to 262144 before timing
        self.growth = list(self.cache.growth_log)
        kb.dispose()
        vb.dispose()
        # one bulk append of the whole history into another layer: the append roofline sample
        self.bulk_k = upload(device, k_all[:context])
        self.bulk_v = upload(device, v_all[:context])
        self.bulk_layer = engine.Int8KvLayer(device, context)
        self.q = upload(device, synthetic(rng, (steps, 16, 256)))
        self.k_new = upload(device, k_all[context:context + steps])
        self.v_new = upload(device, v_all[context:context + steps])
        self.gate = upload(device, synthetic(rng, (steps, 16, 256)))
        self.rotated = device.allocate(steps * 16384)
        self.out = device.allocate(steps * 16384)
        self.pos0 = context

    def run(self):
        """One command of `steps` tokens; each token appends to and attends over every layer.
        The positions advance from run to run (capacity was grown for all of them)."""
        d = self.device
        d.begin()
        for i in range(self.steps):
            pos = self.pos0 + i
            for layer in self.cache.layers:
                # batch_rope_int8 (M = 1) + attention over keys 0..pos, in one dispatch
                engine.decode_append(d, layer, self.q.at(i * 16384), self.k_new.at(i * 2048), self.v_new.at(i * 2048),
                                     self.rotated.at(i * 16384), self.gate.at(i * 16384), self.out.at(i * 16384), pos)
        d.end()

    def bulk_append(self):
        d = self.device
        d.begin()
        engine.store_rows(d, self.bulk_layer, self.bulk_k, self.bulk_v, self.context, 0)
        d.end()

    def kv_bytes(self):
        # 1040 B per attended token and layer: 512 K + 512 V codes + 8 + 8 scale bytes (both KV heads)
        return len(self.cache.layers) * sum(1040 * (self.pos0 + i + 1) for i in range(self.steps))


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-decode", action="store_true")
    ap.add_argument("--no-reference-shapes", action="store_true",
                    help="skip the timings at the reference's kernel shapes (profiling runs: the attention "
                         "kernel's launches are then config 3's chunks only)")
    ap.add_argument("--decode-steps", type=int, default=256,
                    help="decode tokens per timed run (each over every layer); the counter runs "
                         "of the profiles use fewer: traffic per launch does not depend on it")
    ap.add_argument("--copy-probe", action="store_true",
                    help="only run three 1 GiB device-to-device copies (boot_copy): the known-size "
                         "reference that scales rocprofv3 FETCH_SIZE / WRITE_SIZE into bytes")
    args = ap.parse_args()
    if args.gpus != 1:
        print(json.dumps({"error": "this build runs on one GPU; sharding the KV path across GPUs (by KV head, "
                                   "layer or sequence range) is a design, not built",
                          "n_gpus": args.gpus}))
        sys.exit(2)

    device = Device()
    if args.copy_probe:
        n = 1 << 30
        a, b = device.allocate(n), device.allocate(n)
        for _ in range(3):
            device.copy(b, 0, a, 0, n)
        print(json.dumps({"copy_probe_bytes": n, "copies": 3}), flush=True)
        device.close()
        return
    # ---- uninstrumented timed loops first: once wall accounting is reset (below), it
    # stays on for the rest of the context's life
    work = PrefillWorkload(device)
    for _ in range(args.warmup):
        work.step()
    # each step ends with the library's stream synchronized (boot_end)
    t0 = time.perf_counter()
    for _ in range(args.steps):
        work.step()
    wall_ms = (time.perf_counter() - t0) * 1000.0 / args.steps
    control = Fp16ControlWorkload(work)
    for _ in range(args.warmup):
        control.step()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        control.step()
    fp16_ms = (time.perf_counter() - t0) * 1000.0 / args.steps
    dec = None
    if not args.no_decode:
        dec = DecodeWorkload(device, steps=args.decode_steps)
        dec.run()  # warm (the positions are re-appended: the cache bytes are the same)
        t0 = time.perf_counter()
        dec.run()
        dec_wall = (time.perf_counter() - t0) * 1000.0 / dec.steps
        dec.bulk_append()

    # ---- the same work again with every kernel of the path timed by events stamped
    # from its own dispatch (no marker packets on the stream): the roofline's durations
    device.reset_wall_timing(kernels_exact=True)
    for _ in range(args.steps):
        work.step()
    timed = kernel_stats(device, PREFILL_INT8_KERNELS)
    attn_kernel = next((k for k in PREFILL_INT8_KERNELS if k in timed), None)
    if attn_kernel is None:
        raise SystemExit("no INT8 prefill attention kernel was timed")
    ks = kernel_stats(device, ["prefill_combine_kernel", "prepare_fused_int8_kernel"])
    y_int8 = work.out.read(np.float32, work.chunk * 4096)     # the last chunk's INT8 output
    attn_ms = sum(ms for ms, _ in timed.values()) / args.steps
    combine_ms = ks.get("prefill_combine_kernel", (0.0, 0))[0] / args.steps
    launches = sum(n for _, n in timed.values()) // args.steps
    flops = work.flops()
    achieved = flops / (attn_ms * 1e-3) / 1e12
    result = {
        "metric": METRIC, "value": round(wall_ms, 4), "unit": "ms/layer", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(wall_ms, 4), "higher_is_better": False, "scaling": "weak",
        "vs_baseline": None, "dtype": "fp16", "data": "synthetic",
        "config": {"workload": "config 3: 30720-token causal prefill of one full-attention layer, 60 chunks of 512, "
                               "INT8 KV (fused preparation with append + online attention), 16 Q / 2 KV heads, d=256",
                   "kv": "int8 + fp32 per-token/head scales", "tokens": 30720, "chunk": 512,
                   "parallelism": "single GPU"},
        "prefill": {"attention_kernel_ms_per_layer": round(attn_ms, 4), "combine_ms_per_layer": round(combine_ms, 4),
                    "prepare_ms_per_layer": round(ks["prepare_fused_int8_kernel"][0] / args.steps, 4),
                    "attention_launches_per_layer": launches,
                    "mfma_fraction_end_to_end": round(flops / (wall_ms * 1e-3) / 1e12 / MFMA_PEAK_TFLOPS, 4)},
        "roofline": {"bound": "mfma", "kernel": f"{attn_kernel} (attention_online_int8_q32_k256_r2)",
                     "achieved": round(achieved, 2), "peak": MFMA_PEAK_TFLOPS, "unit": "TFLOP/s",
                     "frac": round(achieved / MFMA_PEAK_TFLOPS, 4),
                     "traffic": measured_traffic(attn_kernel),
                     "mfma_busy": (measured_counters(attn_kernel) or {}).get("mfma_busy"),
                     "counters": measured_counters(attn_kernel),
                     "flops_per_layer": flops},
    }
    if not args.no_reference_shapes:
        log("reference shapes: (0,33), (8192,2048), (27900,2048)")
        result["reference_shapes"] = reference_shapes(work)
    device.reset_wall_timing(kernels_exact=True)
    for _ in range(args.steps):
        control.step()
    kc = kernel_stats(device, ["prefill_w64_fp16_kernel", "prefill_combine_kernel", "prepare_fused_half_kernel"])
    y_fp16 = work.out.read(np.float32, work.chunk * 4096)     # the FP16-KV control's, same query and raw K/V
    diff = y_int8.astype(np.float64) - y_fp16
    result["fp16_kv_control"] = {
        "ms_per_layer": round(fp16_ms, 4),
        "kernel": "prefill_w64_fp16_kernel (the INT8 kernel's schedule with FP16 staging)",
        "attention_kernel_ms_per_layer": round(kc.get("prefill_w64_fp16_kernel", (0.0, 0))[0] / args.steps, 4),
        "combine_ms_per_layer": round(kc.get("prefill_combine_kernel", (0.0, 0))[0] / args.steps, 4),
        "prepare_ms_per_layer": round(kc["prepare_fused_half_kernel"][0] / args.steps, 4),
        "int8_over_fp16_time": round(wall_ms / fp16_ms, 4),
        "int8_vs_fp16_output": {"chunk": "last (queries 30208-30719)", "max_abs": float(f"{np.abs(diff).max():.4g}"),
                                "rel_l2": float(f"{np.linalg.norm(diff) / np.linalg.norm(y_fp16):.4g}"),
                                "what": "INT8-cache output minus FP16-cache output of the GPU paths (the quantization "
                                        "error max_abs_quantization_vs_fp16 of Int8KvTests.cs:138-150, measured on "
                                        "the kernels' outputs)"},
        "kv_bytes_30k": {"int8_with_scales": 30720 * 1040, "fp16": 30720 * 2048}}
    if dec is not None:
        device.reset_wall_timing(kernels_exact=True)
        dec.run()
        kd = kernel_stats(device, ["decode_int8_kernel", "decode_combine_kernel"])
        dispatches = dec.steps * len(dec.cache.layers)
        dec_kernel_ms = kd["decode_int8_kernel"][0] / dispatches
        dec_comb_ms = kd.get("decode_combine_kernel", (0.0, 0))[0] / dispatches
        bytes_per_dispatch = dec.kv_bytes() / dispatches
        device.reset_wall_timing(kernels_exact=True)
        dec.bulk_append()
        bulk = kernel_stats(device, ["kv_store_int8_kernel"])["kv_store_int8_kernel"][0]
        bulk_bytes = 5136.0 * dec.context
        result["decode"] = {
            "context": dec.context, "layers": len(dec.cache.layers), "steps": dec.steps, "growth": dec.growth,
            "kv_read_gbs_step": round(dec.kv_bytes() / dec.steps / (dec_wall * 1e-3) / 1e9, 1),
            "kv_read_gbs_attention_kernels": round(bytes_per_dispatch / ((dec_kernel_ms + dec_comb_ms) * 1e-3) / 1e9, 1),
            "ms_per_token_step_wall": round(dec_wall, 5), "decode_kernel_us": round(dec_kernel_ms * 1000, 3),
            "combine_kernel_us": round(dec_comb_ms * 1000, 3),
            "append": "fused into decode_int8_kernel (attention_decode_append_int8)",
            "bytes_per_layer_step": bytes_per_dispatch,
        }
        result["roofline_decode"] = {
            "bound": "hbm", "kernel": "decode_int8_kernel (attention_decode_int8)",
            "achieved": round(bytes_per_dispatch / (dec_kernel_ms * 1e-3) / 1e9, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
            "frac": round(bytes_per_dispatch / (dec_kernel_ms * 1e-3) / 1e9 / HBM_PEAK_GBS, 4),
            "traffic": measured_traffic("decode_int8_kernel"),
            "counters": measured_counters("decode_int8_kernel")}
        result["roofline_append"] = {
            "bound": "hbm", "kernel": "kv_store_int8 bulk append of 131072 tokens",
            "achieved": round(bulk_bytes / (bulk * 1e-3) / 1e9, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
            "frac": round(bulk_bytes / (bulk * 1e-3) / 1e9 / HBM_PEAK_GBS, 4),
            "traffic": measured_traffic("kv_store_int8 bulk 131072"),
            "bytes": bulk_bytes, "kernel_ms": round(bulk, 4)}
    if dec is not None:
        log("verify block and scalar reader: 8 rows at the end of config 4's cache")
        result["verify_block"] = verify_block(dec)
        result["verify_reader"] = verify_reader(dec)
    if not args.no_cpu_baseline:
        log("cpu baseline: the FP64 checker on configs 1, 2, a 131072 decode step and config 3's last chunk")
        result["cpu_baseline"], result["parity_last_chunk"] = cpu_baseline(work, dec, y_int8)
    print(json.dumps(result), flush=True)
    device.close()


if __name__ == "__main__":
    main()
