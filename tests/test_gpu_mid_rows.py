"""Projections with bf16 weights over a middling number of rows (gemm_mid: 128 x 128 tiles, key slices), against numpy in
64 bits and the CPU oracle: partial row and column blocks, widths that are no multiple of 16, every epilogue."""
import numpy as np
import pytest

import ctorch_amd as ct
import oracle
from common import build_pair, say

pytestmark = pytest.mark.gpu
GPU = ct.device("gpu")


# the activations are hi + lo bf16 parts (2^-17 of each), the products f32 sums of at most 2 K roundings of 2^-24
def bound(k):
    return 2.0**-17 + 2 * k * 2.0**-24


@pytest.mark.parametrize("rows,k,n,bias", [(65, 64, 16, False), (65, 512, 17, True), (128, 256, 250, False),
                                           (129, 2048, 48, True), (200, 2048, 2048, False), (256, 64, 33, False),
                                           (300, 4096, 1000, True), (1013, 512, 640, False), (700, 320, 8191, False)])
def test_linear_over_middling_rows(rows, k, n, bias):
    say(f"case: bf16 linear {rows} x {k} -> {n} bias {bias}")
    rng = np.random.default_rng(rows + n)
    x, w, b = (rng.standard_normal(s).astype(np.float32) for s in ((rows, k), (n, k), (n,)))
    wb = oracle.bf16_encode(w)
    w = oracle.bf16_decode(wb)
    got = ct.linear(ct.Tensor.from_numpy(x, ct.F32, GPU), ct.Tensor.from_numpy(wb, ct.BF16, GPU),
                    ct.Tensor.from_numpy(b, ct.F32, GPU) if bias else None).numpy()
    want = x.astype(np.float64) @ w.T.astype(np.float64) + (b if bias else 0.0)
    scale = np.abs(x).astype(np.float64) @ np.abs(w).T.astype(np.float64) + np.abs(want)
    assert np.all(np.abs(got - want) <= bound(k) * scale)


def test_linear_keeps_nans_to_their_rows_and_columns():
    say("case: bf16 linear with a NaN activation and a NaN weight row beside a partial tile")
    rng = np.random.default_rng(3)
    x, w = rng.standard_normal((70, 128)).astype(np.float32), rng.standard_normal((41, 128)).astype(np.float32)
    x[66, 3], w[40, 7] = np.nan, np.nan
    got = ct.linear(ct.Tensor.from_numpy(x, ct.F32, GPU), ct.Tensor.from_numpy(oracle.bf16_encode(w), ct.BF16, GPU)).numpy()
    want = np.zeros((70, 41), bool)
    want[66], want[:, 40] = True, True
    assert np.array_equal(np.isnan(got), want)


@pytest.mark.parametrize("batch,length,d,heads,kv,hidden,rank,kv_dtype", [
    (1, 65, 256, 4, 2, 512, 0, None), (1, 200, 512, 8, 2, 1408, 16, None), (3, 77, 512, 8, 8, 528, 0, ct.BF16),
    (2, 150, 256, 8, 2, 512, 8, None), (70, 1, 256, 4, 2, 512, 0, None)])
def test_prompts_of_middling_length_match_the_oracle(batch, length, d, heads, kv, hidden, rank, kv_dtype):
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
    for part in (ids, ids[:, :1], ids[:, :1]):  # the prompt, then steps over the keys and values that it stored
        want = ref.logits(part, rc)[:, -1]
        assert np.max(np.abs(gpu.logits(part, gc) - want)) <= 2e-2


@pytest.mark.parametrize("rows", [65, 128, 200, 513])
def test_swiglu_block_over_middling_rows(rows):
    say(f"case: SwiGLU module, {rows} rows, 512 -> 1408")
    rng = np.random.default_rng(rows)
    x = rng.standard_normal((rows, 512)).astype(np.float32)
    out = ct.C.c_void_p()
    ct.check(ct.lib().dl_swiglu_create(512, 1408, 0, ct.options(ct.BF16), ct.C.byref(out)))
    block = ct.Module(out)
    bits = {name: oracle.bf16_encode((0.05 * rng.standard_normal(t.shape)).astype(np.float32))
            for name, t in block.state().items()}
    block.load_state(bits, {name: ct.BF16 for name in bits})
    w = {name.split(".")[0]: oracle.bf16_decode(v).astype(np.float64) for name, v in bits.items()}
    gate, up = x @ w["gate"].T, x @ w["up"].T
    want = (gate / (1.0 + np.exp(-gate)) * up) @ w["down"].T
    got = block.forward(ct.Tensor.from_numpy(x, ct.F32, GPU)).numpy()
    assert np.linalg.norm(got - want) <= 2e-5 * np.linalg.norm(want)
