#!/usr/bin/env python3
"""Decode throughput of the MI355X decoder token loop (decode tok/s, 1B bf16, b=1 and b=32,
plus achieved HBM GB/s against the MI355X peak).

Workload of `value` ("C2"): 1B-class GQA decoder (vocab 32000, d 2048, 16 layers, 32/8 heads,
head dim 64, SwiGLU 5632, RoPE base 10000), bf16 weights with f32 accumulation, batch 1, seeded N(0, 0.02) weights
synthesised in HBM, a 128-token prompt of uniform random ids, greedy decode.  A step is one full token step on
the GPU: embedding gather -> 16 fused layers -> final norm + LM head -> sampling -> id fed back, replayed from a
HIP graph; exactly --steps steps are timed with HIP events on the library's compute stream after --warmup
untimed steps.

Also reported: the same C2 decode with temperature-1.0 sampling under an explicit key,
the b=32 decode over a 2048-token seeded K/V prefix ("C3"), the 8B-class b=8 decode over
a 32768-token seeded K/V prefix ("C4"), the per-kernel roofline of
the dominant kernel (gate/up projection: each layer's launch repeated back to back between two HIP events on the
compute stream), a streaming-copy bandwidth reference, and the CPU oracle timed on this host (single thread) on
a bounded sample of the same workload.
"""
import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBPS = 8000.0
# HBM bytes per launch of the gate/up kernel: rocprofv3 --pmc FETCH_SIZE and WRITE_SIZE per dispatch, each scaled
# by what the counter reads for this script's 1 GiB copy probe (x2.0 and x1.0); the commands and the table are in
# the traffic summary under profiles/.  A measurement of the kernel as built, not derived from the bytes below.
GATE_UP_TRAFFIC_BYTES = 46_372_045 + 45_056
C2 = dict(vocab=32000, layers=16, dimensions=2048, heads=32, kv_heads=8, hidden=5632)
C4 = dict(vocab=32000, layers=32, dimensions=4096, heads=32, kv_heads=8, hidden=14336, rope_base=500000.0)
C5 = dict(C2, lora_rank=16, lora_alpha=32.0)
C1 = dict(vocab=256, layers=4, dimensions=256, heads=8, kv_heads=2, hidden=688)
MFMA_BF16_PEAK_TFLOPS = 2500.0


def log(msg):
    print(msg, file=sys.stderr, flush=True)


def parameter_slots(cfg):
    """LM wrapper parameter order (registration order): tokens, decoder layers, final norm, output head."""
    d, H, KV, F, V = cfg["dimensions"], cfg["heads"], cfg["kv_heads"], cfg["hidden"], cfg["vocab"]
    hd = d // H
    names = [("tokens.weight", (V, d))]
    for i in range(cfg["layers"]):
        p = f"decoder.layer{i}."
        names += [(p + "attention.query.weight", (H * hd, d)), (p + "attention.key.weight", (KV * hd, d)),
                  (p + "attention.value.weight", (KV * hd, d)), (p + "attention.output.weight", (d, H * hd))]
        if cfg.get("lora_rank"):
            r = cfg["lora_rank"]
            names += [(p + "attention.query_adapter.down.weight", (r, d)),
                      (p + "attention.query_adapter.up.weight", (H * hd, r)),
                      (p + "attention.value_adapter.down.weight", (r, d)),
                      (p + "attention.value_adapter.up.weight", (KV * hd, r))]
        names += [(p + "feedforward.gate.weight", (F, d)), (p + "feedforward.up.weight", (F, d)),
                  (p + "feedforward.down.weight", (d, F)), (p + "attention_norm.weight", (d,)),
                  (p + "feedforward_norm.weight", (d,))]
    names += [("decoder.normalization.weight", (d,)), ("output.weight", (V, d))]
    return names


def build_model(ct, cfg, context, root=(1234, 0), dtype=None, kv_dtype=None):
    """Seeded weights drawn directly in HBM: slot s gets 0.02 * randn(fold_in(root, s)) rounded to bf16 (LoRA up
    matrices 1e-3 * randn); unmerged LoRA adapters on q and v when cfg has lora_rank.  The K/V cache is f32 (the
    reference's dtype) unless kv_dtype asks for bf16."""
    gpu = ct.device("gpu")
    dtype = ct.BF16 if dtype is None else dtype
    decoder = ct.transformer_decoder(cfg["layers"], cfg["dimensions"], cfg["heads"], cfg["kv_heads"], cfg["hidden"],
                                     context, dtype, gpu, cfg.get("rope_base", 10000.0), kv_dtype=kv_dtype)
    if cfg.get("lora_rank"):
        ct.check(ct.lib().dl_transformer_decoder_attach_lora(decoder.handle, cfg["lora_rank"], cfg["lora_alpha"], 1, 1))
    state, embedding, head = {}, None, None
    for slot, (name, shape) in enumerate(parameter_slots(cfg)):
        if name.endswith("norm.weight") or name == "decoder.normalization.weight":
            continue  # RMSNorm weights keep their module default (ones)
        scale = 1e-3 if name.endswith("_adapter.up.weight") else 0.02
        w = ct.normal(ct.fold_in(root, slot), shape, scale, dtype, gpu)
        if name == "tokens.weight":
            embedding = w
        elif name == "output.weight":
            head = w
        else:
            state[name[len("decoder."):]] = w
    current = decoder.state()
    for name, tensor in current.items():
        state.setdefault(name, tensor)
    decoder.load_state(state)
    del state, current
    lm = ct.DecoderLM(ct.embedding_from(embedding), decoder, ct.linear_from(head))
    return decoder, lm


def weight_bytes(cfg):
    d, H, KV, F, V = cfg["dimensions"], cfg["heads"], cfg["kv_heads"], cfg["hidden"], cfg["vocab"]
    hd = d // H
    per_layer = (H * hd + 2 * KV * hd) * d + d * H * hd + 3 * F * d
    return 2 * (cfg["layers"] * per_layer + V * d)  # LM head once; one embedding row per sequence is negligible


def kv_bytes(cfg, batch, length, element=4):
    """K and V read per step: f32 (4 bytes) for the reference's cache dtype, 2 for the bf16 opt-in."""
    hd = cfg["dimensions"] // cfg["heads"]
    return element * batch * cfg["layers"] * 2 * cfg["kv_heads"] * hd * length


SAMPLE_KEY = (2024, 7)  # the explicit random key of the sampled C2 leg


def decode_b1(ct, steps, warmup):
    context = 128 + 3 + warmup + steps + 8
    decoder, lm = build_model(ct, C2, max(384, context))
    prompt = np.random.default_rng(7).integers(0, C2["vocab"], size=(1, 128), dtype=np.int64)
    cache = ct.DecoderCache(decoder)
    ms, tokens = lm.benchmark(prompt, cache, warmup, steps, 0.0, (0, 0), True)
    # the same decode with temperature-1.0 explicit-key sampling (C2's second leg), on a fresh cache
    scache = ct.DecoderCache(decoder)
    sampled_ms, _ = lm.benchmark(prompt, scache, warmup, steps, 1.0, SAMPLE_KEY, True)
    del scache
    # mean cache length over the timed steps: prompt + tokens before them, + the step's own key
    first = 128 + 3 + warmup
    mean_len = first + (steps - 1) / 2.0
    step_bytes = weight_bytes(C2) + kv_bytes(C2, 1, mean_len)
    # per-kernel-class device time: each class's launches of one step (one per layer) repeated back to back
    # between two HIP events on the compute stream (cold weights: a class's 16 layers exceed the 256 MB cache)
    pcache = ct.DecoderCache(decoder)
    lm.logits(prompt, pcache)
    timings = lm.profile(prompt[:, -1:], pcache, 10)
    return dict(ms=ms, sampled_ms=sampled_ms, step_bytes=step_bytes, timings=timings, tokens=tokens,
                mean_len=mean_len), decoder, lm


def decode_b32(ct, steps, warmup, prefix=2048):
    """C3: batch 32, each sequence holding `prefix` cached tokens of seeded random K/V in the bf16 cache opt-in
    (the KV-bandwidth regime, sized in bf16)."""
    B = 32
    decoder, lm = build_model(ct, C2, prefix + 3 + warmup + steps + 8, kv_dtype=ct.BF16)
    cache = ct.DecoderCache(decoder)
    hd = C2["dimensions"] // C2["heads"]
    for layer in range(C2["layers"]):
        k = ct.normal(ct.fold_in((4242, 0), 2 * layer), [B, C2["kv_heads"], prefix, hd], 1.0, ct.BF16)
        v = ct.normal(ct.fold_in((4242, 0), 2 * layer + 1), [B, C2["kv_heads"], prefix, hd], 1.0, ct.BF16)
        cache.append(layer, k, v)
        del k, v
    ids = np.random.default_rng(8).integers(0, C2["vocab"], size=(B, 1), dtype=np.int64)
    ms, _ = lm.benchmark(ids, cache, warmup, steps, 0.0, (0, 0), True)
    mean_len = prefix + 3 + warmup + (steps - 1) / 2.0
    return dict(ms=ms, step_bytes=weight_bytes(C2) + kv_bytes(C2, B, mean_len, 2), batch=B, mean_len=mean_len)


def decode_c4(ct, steps, warmup, batch=8, prefix=32768):
    """C4: the 8B-class decoder (RoPE base 500000), batch 8, each sequence holding `prefix` cached positions of
    seeded random K/V (34 GB in the bf16 cache opt-in at 32768), greedy decode."""
    cfg = C4
    decoder, lm = build_model(ct, cfg, prefix + 3 + warmup + steps + 8, root=(88, 0), kv_dtype=ct.BF16)
    cache = ct.DecoderCache(decoder)
    hd = cfg["dimensions"] // cfg["heads"]
    for layer in range(cfg["layers"]):
        k = ct.normal(ct.fold_in((4343, 0), 2 * layer), [batch, cfg["kv_heads"], prefix, hd], 1.0, ct.BF16)
        v = ct.normal(ct.fold_in((4343, 0), 2 * layer + 1), [batch, cfg["kv_heads"], prefix, hd], 1.0, ct.BF16)
        cache.append(layer, k, v)
        del k, v
    ids = np.random.default_rng(9).integers(0, cfg["vocab"], size=(batch, 1), dtype=np.int64)
    ms, _ = lm.benchmark(ids, cache, warmup, steps, 0.0, (0, 0), True)
    mean_len = prefix + 3 + warmup + (steps - 1) / 2.0
    return dict(ms=ms, step_bytes=weight_bytes(cfg) + kv_bytes(cfg, batch, mean_len, 2), batch=batch, mean_len=mean_len)


def prefill_flops(cfg, batch, length):
    """Algorithmic FLOPs of a prefill chunk: 2 * (decoder linear + LoRA parameters) per token, causal QK^T and PV
    (4 * hd per visible query-key pair), and the LM head on the last position of each sequence."""
    d, H, KV, F, V = cfg["dimensions"], cfg["heads"], cfg["kv_heads"], cfg["hidden"], cfg["vocab"]
    hd = d // H
    linear = (H * hd + 2 * KV * hd) * d + d * H * hd + 3 * F * d
    if cfg.get("lora_rank"):
        r = cfg["lora_rank"]
        linear += r * d + H * hd * r + r * d + KV * hd * r
    pairs = length * (length + 1) / 2
    return (2.0 * cfg["layers"] * linear * batch * length + 4.0 * cfg["layers"] * batch * H * hd * pairs
            + 2.0 * batch * V * d)


def prefill_c5(ct, decode_steps, batch=4, length=4096):
    """C5: the 1B-class decoder with unmerged LoRA (r=16, alpha=32) on q and v; prefill of `batch` x `length`
    uniform random ids (timed with HIP events on the compute stream, after one untimed prefill), then greedy
    decode of `decode_steps` tokens from the HIP graph."""
    decoder, lm = build_model(ct, C5, length + decode_steps + 16, root=(555, 0))
    prompt = np.random.default_rng(10).integers(0, C5["vocab"], size=(batch, length), dtype=np.int64)
    cache = ct.DecoderCache(decoder)
    lm.logits(prompt, cache)  # untimed: workspaces, first-touch
    cache.truncate(0)
    timer = ct.Timer()
    timer.start()
    logits = lm.logits(prompt, cache)
    prefill_ms = timer.stop()
    ids = logits.argmax(-1).reshape(batch, 1).astype(np.int64)
    ms = 0.0
    if decode_steps > 0:  # --c5-steps 0: the prefill alone
        ms, _ = lm.benchmark(ids, cache, 2, decode_steps, 0.0, (0, 0), True)
    flops = prefill_flops(C5, batch, length)
    mean_len = length + 3 + (decode_steps - 1) / 2.0
    return dict(prefill_ms=prefill_ms, flops=flops, decode_ms=ms, batch=batch, length=length,
                step_bytes=weight_bytes(C5) + kv_bytes(C5, batch, mean_len))


def decode_c1(ct, steps=128, prompt_len=32):
    """C1: the tiny f32 decoder (byte vocabulary), a 32-byte prompt then `steps` greedy steps from the HIP graph
    (launch-bound: 11 MB of weights sit in the Infinity Cache; reported as an absolute number)."""
    decoder, lm = build_model(ct, C1, 192, root=(11, 0), dtype=ct.F32)
    prompt = np.random.default_rng(11).integers(0, C1["vocab"], size=(1, prompt_len), dtype=np.int64)
    ms, _ = lm.benchmark(prompt, ct.DecoderCache(decoder), 0, steps - 1, 0.0, (0, 0), True)
    return dict(ms=ms, steps=steps - 1)


def host_cpu():
    """The host's CPU model (from /proc/cpuinfo) and its logical CPU count."""
    model = "unknown"
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    return model, os.cpu_count() or 1


def cpu_baseline(threads=16):
    """The CPU oracle (plain-C restatement of the reference CPU path) on this host, per the plan of the reference's
    CPU path: single-threaded as the reference's CPU kernels are, and, for the legs whose single-thread time would
    run for minutes, a labelled row-parallel variant (bit-identical results) on `threads` threads.

      C1  the tiny f32 decoder in full: 32-byte prompt, then 128 greedy steps (1 thread);
      C2  1B bf16: the 128-token prompt (untimed setup, all threads), then 16 greedy decode steps timed (1 thread);
      C3  1B bf16 at batch 32 over a 2048-token seeded prefix: 2 decode steps timed (`threads` threads);
      C4  8B-width: 8 decode steps of one layer at batch 8 over a 32768-position prefix, timed on `threads`
          threads and reported for the 32-layer model as 32 x that time (embedding and LM head not timed);
      C5  1B bf16 + LoRA r16: a 1 x 512 prefill sample timed (`threads` threads).
    Weights are synthesised on the host with all threads before each leg (untimed)."""
    import oracle
    oracle.lib()
    threads = max(1, min(threads, os.cpu_count() or 1))
    model, nproc = host_cpu()
    legs = {}

    def lm_for(cfg, root):
        oracle.set_threads(threads)
        return oracle.OracleLM(cfg, oracle.synthesize_weights(cfg, root))

    def timed(fn, n_threads):
        oracle.set_threads(n_threads)
        t0 = time.perf_counter()
        out = fn()
        return out, time.perf_counter() - t0

    # C1
    c1 = oracle.ModelConfig(vocab=256, layers=4, dimensions=256, heads=8, kv_heads=2, hidden=688, context=168,
                            dtype="f32")
    lm = lm_for(c1, (11, 0))
    prompt = np.random.default_rng(11).integers(0, 256, size=(1, 32), dtype=np.int64)
    _, sec = timed(lambda: lm.generate(prompt, 128), 1)
    legs["c1"] = dict(value=128 / sec, unit="tok/s", cores=1, seconds=sec,
                      sample="C1 in full: 32-byte prompt + 128 greedy steps (prompt included in the time)")
    # C2
    c2 = oracle.ModelConfig(vocab=32000, layers=16, dimensions=2048, heads=32, kv_heads=8, hidden=5632, context=160,
                            dtype="bf16")
    lm = lm_for(c2, (1234, 0))
    cache = lm.make_cache(1)
    prompt = np.random.default_rng(7).integers(0, c2.vocab, size=(1, 128), dtype=np.int64)
    oracle.set_threads(threads)
    token = lm.logits(prompt, cache)[:, -1].argmax(-1).reshape(1, 1)

    def c2_steps():
        t = token
        for _ in range(16):
            t = lm.logits(t, cache)[:, -1].argmax(-1).reshape(1, 1)
    _, sec = timed(c2_steps, 1)
    legs["c2"] = dict(value=16 / sec, unit="tok/s", cores=1, seconds=sec,
                      sample="C2: 128-token prompt (untimed), then 16 greedy decode steps at cache lengths 128-143")
    # C3: the same 1B weights, batch 32 over a seeded 2048-token prefix (bf16-exact values, one block per layer)
    B, P = 32, 2048
    lm3 = oracle.OracleLM(oracle.ModelConfig(**{**c2.__dict__, "context": P + 4}), lm.w)
    cache = lm3.make_cache(B)
    n = B * c2.kv_heads * P * c2.head_dim
    kv = [oracle.bf16_decode(oracle.bf16_encode(oracle.randn(oracle.fold_in((4242, 0), j), n)))
          .reshape(B, c2.kv_heads, P, c2.head_dim) for j in (0, 1)]
    for layer in range(c2.layers):
        cache.fill(layer, P, kv[0], kv[1])
    del kv
    ids = np.random.default_rng(8).integers(0, c2.vocab, size=(B, 1), dtype=np.int64)

    def c3_steps():
        t = ids
        for _ in range(2):
            t = lm3.logits(t, cache)[:, -1].argmax(-1).reshape(B, 1)
    _, sec = timed(c3_steps, threads)
    legs["c3"] = dict(value=2 * B / sec, unit="tok/s", cores=threads, seconds=sec,
                      sample="C3: batch 32 over a 2048-token seeded prefix, 2 greedy decode steps (row-parallel)")
    del cache, lm3, lm
    # C4: one layer of the 8B-width decoder (its weights only: a 16-entry vocabulary keeps the embedding and the
    # head out of the way), 8 decode steps at batch 8 over a 32768-position prefix, each reported for the 32
    # layers of the model.  The prefix holds constants, written to every page of the cache (the arithmetic's time does not depend
    # on the values, and drawing 2 x 268M random values would cost a minute)
    c4 = oracle.ModelConfig(vocab=16, layers=1, dimensions=4096, heads=32, kv_heads=8, hidden=14336,
                            context=32768 + 16, dtype="bf16", rope_base=500000.0)
    lm4 = lm_for(c4, (88, 0))
    B4, P4 = 8, 32768
    cache = lm4.make_cache(B4)
    cache.keys[0][:, :, :P4] = 0.25
    cache.values[0][:, :, :P4] = -0.5
    cache.structs[0].length = P4
    x4 = np.random.default_rng(12).standard_normal((B4, 1, c4.dimensions), dtype=np.float32)
    def c4_steps():
        for _ in range(8):
            lm4.decode(x4, cache)
    _, sec = timed(c4_steps, threads)
    legs["c4"] = dict(value=8 * B4 / (32 * sec), unit="tok/s", cores=threads, seconds=sec, layers_timed=1,
                      sample="C4: 8 decode steps of one 8B-width layer (d 4096, 32/8 heads, head dim 128, SwiGLU "
                             "14336) at batch 8 over 32768-32775 cached positions, reported as 32 x the layer "
                             "time (embedding and LM head not timed; row-parallel)")
    del cache, lm4
    # C5
    c5 = oracle.ModelConfig(vocab=32000, layers=16, dimensions=2048, heads=32, kv_heads=8, hidden=5632, context=520,
                            dtype="bf16", lora_rank=16, lora_alpha=32.0)
    lm = lm_for(c5, (555, 0))
    prompt = np.random.default_rng(10).integers(0, c5.vocab, size=(1, 512), dtype=np.int64)
    cache = lm.make_cache(1)
    _, sec = timed(lambda: lm.logits(prompt, cache), threads)
    legs["c5"] = dict(value=512 / sec, unit="tok/s", cores=threads, seconds=sec,
                      sample="C5: prefill of 1 x 512 tokens with unmerged LoRA r16 (row-parallel)")
    c2leg = legs["c2"]
    return dict(value=c2leg["value"], unit="tok/s", cores=1, kind="port",
                sample=f"1B bf16 b=1 (C2): 128-token prompt then 16 greedy decode steps timed ({c2leg['seconds']:.1f} s), "
                       f"oracle/oracle.c -O3 -ffp-contract=off, 1 thread",
                cpu_model=model, nproc=nproc, legs=legs)


def main():
    ap = argparse.ArgumentParser(description=__doc__.split("\n")[0])
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=256)
    ap.add_argument("--warmup", type=int, default=16)
    ap.add_argument("--b32-steps", type=int, default=32)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-b32", action="store_true")
    ap.add_argument("--c4-steps", type=int, default=16)
    ap.add_argument("--no-c4", action="store_true")
    ap.add_argument("--c5-steps", type=int, default=128)
    ap.add_argument("--no-c5", action="store_true")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py measures one GPU: this build has no multi-GPU path (asked for --gpus {args.gpus})",
              file=sys.stderr)
        sys.exit(2)

    import ctorch_amd as ct
    ct.lib()
    log("bench: copy bandwidth probe")
    copy_gbps = ct.copy_bandwidth(1 << 30, 20)
    log(f"bench: streaming copy {copy_gbps:.0f} GB/s; building 1B bf16 model in HBM")
    b1, decoder, lm = decode_b1(ct, args.steps, args.warmup)
    ms_per_step = b1["ms"] / args.steps
    tok_s = args.steps / (b1["ms"] / 1e3)
    achieved = b1["step_bytes"] / (ms_per_step / 1e3) / 1e9
    log(f"bench: b=1 {ms_per_step * 1e3:.1f} us/step, {tok_s:.0f} tok/s, {achieved:.0f} GB/s algorithmic")
    sampled_us = 1e3 * b1["sampled_ms"] / args.steps
    log(f"bench: b=1 temperature 1.0 (explicit key) {sampled_us:.1f} us/step, {1e6 / sampled_us:.0f} tok/s")

    gate = next(t for t in b1["timings"] if t["name"] == "gate_up_silu")
    gate_avg_ms = gate["total_ms"] / gate["launches"]
    gate_bytes = gate["bytes"] / gate["launches"]
    gate_gbps = gate_bytes / (gate_avg_ms / 1e3) / 1e9
    kernels = {t["name"]: {"launches": t["launches"], "avg_us": 1e3 * t["total_ms"] / t["launches"],
                           "GB/s": (t["bytes"] / t["total_ms"] * 1e-6) if t["total_ms"] > 0 and t["bytes"] else None}
               for t in b1["timings"]}

    extra = {"c2_sampled": {"tok_s": 1e6 / sampled_us, "us_per_step": sampled_us, "temperature": 1.0,
                            "key": list(SAMPLE_KEY), "steps": args.steps, "warmup": args.warmup}}
    c1 = decode_c1(ct)
    extra["c1"] = {"tok_s": c1["steps"] / (c1["ms"] / 1e3), "us_per_step": 1e3 * c1["ms"] / c1["steps"],
                   "steps": c1["steps"], "prompt": 32, "dtype": "f32"}
    log(f"bench: C1 {extra['c1']['us_per_step']:.1f} us/step, {extra['c1']['tok_s']:.0f} tok/s")
    del lm, decoder  # free the C2 model's HBM before the larger workloads
    import gc
    gc.collect()
    if not args.no_b32:
        log("bench: b=32 over a 2048-token prefix")
        b32 = decode_b32(ct, args.b32_steps, 4)
        ms32 = b32["ms"] / args.b32_steps
        extra["b32"] = {"tok_s": 32 * args.b32_steps / (b32["ms"] / 1e3), "ms_per_step": ms32,
                        "achieved_GBps": b32["step_bytes"] / (ms32 / 1e3) / 1e9,
                        "frac_of_peak": b32["step_bytes"] / (ms32 / 1e3) / 1e9 / HBM_PEAK_GBPS,
                        "steps": args.b32_steps, "prefix": 2048}
        log(f"bench: b=32 {ms32:.3f} ms/step, {extra['b32']['tok_s']:.0f} tok/s")

    if not args.no_c4:
        log("bench: C4 8B b=8 over a 32768-token prefix")
        gc.collect()
        c4 = decode_c4(ct, args.c4_steps, 2)
        ms4 = c4["ms"] / args.c4_steps
        extra["c4"] = {"tok_s": c4["batch"] * args.c4_steps / (c4["ms"] / 1e3), "ms_per_step": ms4,
                       "achieved_GBps": c4["step_bytes"] / (ms4 / 1e3) / 1e9,
                       "frac_of_peak": c4["step_bytes"] / (ms4 / 1e3) / 1e9 / HBM_PEAK_GBPS,
                       "steps": args.c4_steps, "prefix": 32768, "batch": c4["batch"]}
        log(f"bench: C4 {ms4:.2f} ms/step, {extra['c4']['tok_s']:.0f} tok/s, {extra['c4']['achieved_GBps']:.0f} GB/s")
        del c4

    if not args.no_c5:
        log("bench: C5 prefill 4 x 4096 with LoRA, then decode")
        gc.collect()
        c5 = prefill_c5(ct, args.c5_steps)
        tflops = c5["flops"] / (c5["prefill_ms"] / 1e3) / 1e12
        ms5 = c5["decode_ms"] / max(1, args.c5_steps)
        extra["c5"] = {"prefill_tok_s": c5["batch"] * c5["length"] / (c5["prefill_ms"] / 1e3),
                       "prefill_ms": c5["prefill_ms"], "prefill_TFLOPs": tflops,
                       "mfma_utilisation": tflops / MFMA_BF16_PEAK_TFLOPS, "prefill_flops": c5["flops"],
                       "decode_tok_s": c5["batch"] * args.c5_steps / (c5["decode_ms"] / 1e3) if args.c5_steps > 0 else None,
                       "decode_ms_per_step": ms5 if args.c5_steps > 0 else None,
                       "decode_steps": args.c5_steps, "batch": c5["batch"], "prompt": c5["length"],
                       "lora": "r=16, alpha=32 on q and v (unmerged)"}
        log(f"bench: C5 prefill {c5['prefill_ms']:.1f} ms ({extra['c5']['prefill_tok_s']:.0f} tok/s, "
            f"{tflops:.0f} TFLOP/s), decode {ms5:.3f} ms/step")
        del c5

    baseline = None
    if not args.no_cpu_baseline:
        log("bench: CPU oracle baseline (C1, C2 single thread; C3, C4, C5 row-parallel samples)")
        baseline = cpu_baseline()
        log("bench: CPU " + ", ".join(f"{k} {v['value']:.3g} {v['unit']} ({v['cores']} thr, {v['seconds']:.1f} s)"
                                      for k, v in baseline["legs"].items()) + f" on {baseline['cpu_model']}")

    line = {
        "metric": "decode tok/s (1B bf16, b=1 and b=32) + achieved HBM GB/s vs MI355X peak",
        "value": tok_s,
        "unit": "tok/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms_per_step,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic: seeded N(0,0.02) bf16 weights drawn in HBM, 128 uniform random prompt ids, greedy",
        "config": {"workload": "C2: 1B-class GQA decoder bf16, batch 1, 128-token prompt, greedy decode",
                   "vocab": 32000, "d_model": 2048, "layers": 16, "heads": 32, "kv_heads": 8, "head_dim": 64,
                   "hidden": 5632, "batch": 1, "prompt": 128, "mean_cache_length": b1["mean_len"]},
        "achieved_GBps": achieved,
        "frac_of_hbm_peak": achieved / HBM_PEAK_GBPS,
        "copy_GBps": copy_gbps,
        "roofline": {"bound": "hbm",
                     "kernel": "gemv_reg<bf16, MT=1, R=2, CPI=4, SWIGLU> (RMSNorm + gate/up projection + SiLU*up)",
                     "achieved": gate_gbps, "peak": HBM_PEAK_GBPS, "unit": "GB/s", "frac": gate_gbps / HBM_PEAK_GBPS,
                     "traffic": GATE_UP_TRAFFIC_BYTES, "bytes_per_launch": gate_bytes, "avg_launch_us": gate_avg_ms * 1e3},
        "kernels": kernels,
        "cpu_baseline": baseline,
    }
    line.update(extra)
    print(json.dumps(line))


if __name__ == "__main__":
    main()
