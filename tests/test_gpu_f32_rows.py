"""Projections on the f32 matrix cores, against numpy in 64 bits and the CPU oracle: f32 weights over nine or more rows,
and bf16 weights over 65 or more of the shapes whose activations are not split.  Edges of the work-group shapes, partial
weight tiles, K remainders, every epilogue.  test_host_rules.py checks on the CPU that each shape takes the work-groups named
beside it."""
import numpy as np
import pytest

import ctorch_amd as ct
import oracle
from common import build_pair, rel_err, say

pytestmark = pytest.mark.gpu
GPU = ct.device("gpu")


# 16 k are summed in f32 and the sums of 16 in f64: at most 16 roundings of 2^-24 on each product, and one at the end
BOUND = 17 * 2.0**-24


# rows, k, n, work-group shape
LINEAR_F32 = [(9, 4, 1, "32x16"), (16, 36, 130, "32x16"), (17, 1000, 333, "32x16"), (33, 688, 64, "32x16"),
              (65, 32, 2, "32x16"), (129, 256, 8191, "64x32"), (700, 260, 2100, "64x32"), (2100, 64, 260, "64x32"),
              (1030, 36, 2100, "64x64"), (2049, 36, 8200, "128x128")]


@pytest.mark.parametrize("rows,k,n,shape", LINEAR_F32)
def test_linear_f32_weights_over_many_rows(rows, k, n, shape):
    say(f"case: f32 linear {rows} x {k} -> {n} ({shape})")
    rng = np.random.default_rng(rows)
    x, w, b = (rng.standard_normal(s).astype(np.float32) for s in ((rows, k), (n, k), (n,)))
    gx, gw, gb = (ct.Tensor.from_numpy(a, ct.F32, GPU) for a in (x, w, b))
    scale = np.abs(x).astype(np.float64) @ np.abs(w).T.astype(np.float64)
    for bias, add in ((None, 0.0), (gb, b.astype(np.float64))):
        got = ct.linear(gx, gw, bias).numpy()
        want = x.astype(np.float64) @ w.T.astype(np.float64) + add
        assert np.all(np.abs(got - want) <= BOUND * scale + 2.0**-23 * np.abs(want))


def test_linear_f32_keeps_infinities_and_nans_to_their_rows():
    say("case: f32 linear with an infinite and a NaN activation")
    rng = np.random.default_rng(1)
    x, w = rng.standard_normal((20, 64)).astype(np.float32), np.abs(rng.standard_normal((48, 64))).astype(np.float32)
    x[3, 5], x[7, 60] = np.inf, np.nan
    got = ct.linear(ct.Tensor.from_numpy(x, ct.F32, GPU), ct.Tensor.from_numpy(w, ct.F32, GPU)).numpy()
    assert np.all(np.isposinf(got[3])) and np.all(np.isnan(got[7]))
    assert np.all(np.isfinite(np.delete(got, [3, 7], 0)))


LINEAR_BF16 = [(65, 64, 16, "32x16"), (65, 512, 17, "32x16"), (128, 256, 250, "32x16"), (129, 320, 48, "32x16"),
               (256, 64, 33, "32x16"), (300, 4096, 1000, "32x16"), (300, 320, 8192, "64x64"), (700, 320, 2050, "64x32"),
               (1030, 64, 2100, "64x64"), (2049, 64, 8200, "128x128")]


@pytest.mark.parametrize("rows,k,n,shape", LINEAR_BF16)
def test_linear_bf16_weights_keep_whole_activations(rows, k, n, shape):
    say(f"case: bf16 linear {rows} x {k} -> {n}, f32 activations ({shape})")
    rng = np.random.default_rng(rows + n)
    x, w, b = (rng.standard_normal(s).astype(np.float32) for s in ((rows, k), (n, k), (n,)))
    bits, bias_bits = oracle.bf16_encode(w), oracle.bf16_encode(b)
    w, bias = oracle.bf16_decode(bits), oracle.bf16_decode(bias_bits).astype(np.float64)
    gx, gw = ct.Tensor.from_numpy(x, ct.F32, GPU), ct.Tensor.from_numpy(bits, ct.BF16, GPU)
    scale = np.abs(x).astype(np.float64) @ np.abs(w).T.astype(np.float64)
    dots = x.astype(np.float64) @ w.T.astype(np.float64)
    for gb, add in ((None, 0.0), (ct.Tensor.from_numpy(b, ct.F32, GPU), b.astype(np.float64)),
                    (ct.Tensor.from_numpy(bias_bits, ct.BF16, GPU), bias)):
        got, want = ct.linear(gx, gw, gb).numpy(), dots + add
        assert np.all(np.abs(got - want) <= BOUND * scale + 2.0**-23 * np.abs(want))
        # two bf16 parts of the activations would be off by some 2.5e-6 here
        assert np.linalg.norm(got - want) <= 3e-7 * np.linalg.norm(want)


def test_linear_bf16_weights_keep_infinities_to_their_rows():
    say("case: bf16 linear over 70 rows with an infinite activation")
    rng = np.random.default_rng(2)
    x, w = rng.standard_normal((70, 64)).astype(np.float32), np.abs(rng.standard_normal((48, 64))).astype(np.float32)
    x[66, 5], x[69, 1] = np.inf, np.float32(3.4e38)  # the second is above the largest bf16
    got = ct.linear(ct.Tensor.from_numpy(x, ct.F32, GPU), ct.Tensor.from_numpy(oracle.bf16_encode(w), ct.BF16, GPU)).numpy()
    assert np.all(np.isposinf(got[66])) and np.all(np.isfinite(np.delete(got, [66, 69], 0)))
    assert not np.isnan(got[69]).any()


@pytest.mark.parametrize("rows,d,hidden", [(65, 320, 528), (200, 192, 1008), (1100, 64, 4112)])
def test_swiglu_bf16_weights_keep_whole_activations(rows, d, hidden):
    say(f"case: bf16 SwiGLU module, {rows} rows, {d} -> {hidden}, f32 activations")
    rng = np.random.default_rng(rows)
    x = rng.standard_normal((rows, d)).astype(np.float32)
    out = ct.C.c_void_p()
    ct.check(ct.lib().dl_swiglu_create(d, hidden, 0, ct.options(ct.BF16), ct.C.byref(out)))
    block = ct.Module(out)
    bits = {name: oracle.bf16_encode((0.1 * rng.standard_normal(t.shape)).astype(np.float32))
            for name, t in block.state().items()}
    block.load_state(bits, {name: ct.BF16 for name in bits})
    w = {name.split(".")[0]: oracle.bf16_decode(v).astype(np.float64) for name, v in bits.items()}
    gate, up = x @ w["gate"].T, x @ w["up"].T
    want = (gate / (1.0 + np.exp(-gate)) * up) @ w["down"].T
    got = block.forward(ct.Tensor.from_numpy(x, ct.F32, GPU)).numpy()
    assert np.linalg.norm(got - want) <= 5e-7 * np.linalg.norm(want)


@pytest.mark.parametrize("batch,length,d,heads,kv,hidden,rank,kv_dtype", [
    (1, 65, 320, 10, 2, 528, 0, None), (1, 200, 320, 5, 5, 576, 16, None), (3, 50, 192, 6, 2, 320, 0, ct.BF16),
    (1, 255, 192, 3, 3, 1008, 32, ct.BF16)])
def test_bf16_decoders_of_other_widths_match_the_oracle(batch, length, d, heads, kv, hidden, rank, kv_dtype):
    say(f"case: bf16 decoder, {batch} x {length} positions, d {d}, heads {heads}/{kv}, hidden {hidden}, rank {rank}")
    cfg = oracle.ModelConfig(vocab=97, layers=2, dimensions=d, heads=heads, kv_heads=kv, hidden=hidden,
                             context=length + 4, dtype="bf16", **(dict(lora_rank=rank, lora_alpha=16.0) if rank else {}))
    weights = oracle.synthesize_weights(cfg, (45, 0), 0.05)
    for name in weights:
        if name.endswith("_adapter.up.weight"):
            weights[name] = oracle.bf16_encode(oracle.randn((46, len(name)), weights[name].size) * np.float32(0.1)).reshape(
                weights[name].shape)
    ref, gpu = build_pair(cfg, weights=weights, kv_dtype=kv_dtype)
    ids = oracle.random_ids((47, 0), batch * length, cfg.vocab).reshape(batch, length)
    rc, gc = ref.make_cache(batch), gpu.cache()
    bound = 1e-4 if kv_dtype is None else 2e-2  # the oracle's cache is f32
    for part in (ids, ids[:, :1], ids[:, :1]):  # the prompt, then steps over the keys and values that it stored
        assert rel_err(gpu.logits(part, gc), ref.logits(part, rc)[:, -1]) <= bound


@pytest.mark.parametrize("batch,length,heads,kv,d,hidden,rank,kv_dtype", [
    (1, 9, 4, 2, 32, 36, 0, None), (3, 13, 8, 2, 256, 688, 0, None), (2, 40, 8, 8, 64, 100, 4, None),
    (2, 150, 8, 2, 256, 688, 16, ct.BF16), (1, 700, 8, 2, 256, 688, 8, None)])
def test_decoder_f32_prompts_match_the_oracle(batch, length, heads, kv, d, hidden, rank, kv_dtype):
    say(f"case: f32 decoder, {batch} x {length} positions, d {d}, heads {heads}/{kv}, hidden {hidden}, rank {rank}")
    cfg = oracle.ModelConfig(vocab=97, layers=2, dimensions=d, heads=heads, kv_heads=kv, hidden=hidden,
                             context=length + 4, dtype="f32", **(dict(lora_rank=rank, lora_alpha=8.0) if rank else {}))
    weights = oracle.synthesize_weights(cfg, (77, 0), 0.06)
    for name in weights:
        if name.endswith("_adapter.up.weight"):
            weights[name] = oracle.randn((78, len(name)), weights[name].size).reshape(weights[name].shape) * np.float32(0.1)
    ref, gpu = build_pair(cfg, weights=weights, kv_dtype=kv_dtype)
    ids = oracle.random_ids((79, 0), batch * length, cfg.vocab).reshape(batch, length)
    rc, gc = ref.make_cache(batch), gpu.cache()
    bound = 1e-4 if kv_dtype is None else 2e-2  # the oracle's cache is f32
    assert rel_err(gpu.logits(ids, gc), ref.logits(ids, rc)[:, -1]) <= bound
    # the new positions' keys and values were stored: a step over them agrees too
    ids = ids[:, :1]
    assert rel_err(gpu.logits(ids, gc), ref.logits(ids, rc)[:, -1]) <= bound
