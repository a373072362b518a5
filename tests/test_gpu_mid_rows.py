"""Projections with bf16 weights over 65 rows and more whose activations are split into two bf16 parts (gemm_mid: 128 x 128
tiles, key slices; gemm_tiles: 256 x 256; gemm_narrow), against numpy in 64 bits and the CPU oracle: partial row and column
blocks, every epilogue.  test_host_rules.py checks on the CPU that each shape takes the kernel named beside it."""
import numpy as np
import pytest

import ctorch_amd as ct
import oracle
from common import GpuLM, agree, rel_err, say

pytestmark = pytest.mark.gpu
GPU = ct.device("gpu")


# the activations are hi + lo bf16 parts (2^-17 of each), the products f32 sums of K roundings of 2^-24, of either sign
def bound(k):
    return 2.0**-17 + np.sqrt(k) * 2.0**-24


# rows, k, n, bias, kernel
LINEAR = [(65, 512, 16, True, "mid"), (65, 512, 48, False, "mid"), (128, 768, 256, False, "mid"),
          (129, 2048, 48, True, "mid"), (200, 2048, 2048, False, "mid"), (300, 4096, 1008, True, "mid"),
          (1013, 512, 640, False, "mid"), (700, 768, 8208, False, "mid"), (65, 512, 16, False, "narrow"),
          (300, 1024, 32, False, "narrow"), (333, 512, 32000, False, "tiles"), (333, 512, 32016, True, "tiles"),
          (520, 512, 21008, False, "tiles")]


@pytest.mark.parametrize("rows,k,n,bias,kernel", LINEAR)
def test_linear_over_middling_rows(rows, k, n, bias, kernel):
    say(f"case: bf16 linear {rows} x {k} -> {n} bias {bias} ({kernel})")
    rng = np.random.default_rng(rows + n)
    x, w, b = (rng.standard_normal(s).astype(np.float32) for s in ((rows, k), (n, k), (n,)))
    wb = oracle.bf16_encode(w)
    w = oracle.bf16_decode(wb)
    got = ct.linear(ct.Tensor.from_numpy(x, ct.F32, GPU), ct.Tensor.from_numpy(wb, ct.BF16, GPU),
                    ct.Tensor.from_numpy(b, ct.F32, GPU) if bias else None).numpy()
    want = x.astype(np.float64) @ w.T.astype(np.float64) + (b if bias else 0.0)
    agree(got, want, bound(k))


def test_linear_keeps_nans_to_their_rows_and_columns():
    say("case: bf16 linear with a NaN activation and a NaN weight row beside a partial tile (mid)")
    rng = np.random.default_rng(3)
    x, w = rng.standard_normal((70, 512)).astype(np.float32), rng.standard_normal((48, 512)).astype(np.float32)
    x[66, 3], w[40, 7] = np.nan, np.nan
    got = ct.linear(ct.Tensor.from_numpy(x, ct.F32, GPU), ct.Tensor.from_numpy(oracle.bf16_encode(w), ct.BF16, GPU)).numpy()
    want = np.zeros((70, 48), bool)
    want[66], want[:, 40] = True, True
    assert np.array_equal(np.isnan(got), want)


# batch, length, d, heads, kv, hidden, rank, kv_dtype, kernels of QKV, output, gate/up and down
PROMPTS = [(1, 65, 512, 8, 2, 768, 0, None, "mid, mid, mid, mid"), (1, 200, 512, 8, 2, 1536, 16, None, "mid, mid, mid, mid"),
           (3, 77, 768, 12, 12, 512, 0, ct.BF16, "mid, mid, mid, mid"), (2, 150, 512, 8, 2, 512, 8, None, "mid, mid, mid, mid"),
           (70, 1, 512, 8, 2, 768, 0, None, "mid, mid, mid, mid"), (1, 200, 512, 8, 2, 1408, 16, None, "mid, mid, mid, f32"),
           (3, 77, 512, 8, 8, 528, 0, ct.BF16, "mid, mid, mid, gemv"), (1, 65, 256, 4, 2, 512, 0, None, "f32, f32, f32, mid")]


@pytest.mark.parametrize("batch,length,d,heads,kv,hidden,rank,kv_dtype,kernels", PROMPTS)
def test_prompts_of_middling_length_match_the_oracle(batch, length, d, heads, kv, hidden, rank, kv_dtype, kernels):
    say(f"case: bf16 decoder, {batch} x {length} positions, d {d}, heads {heads}/{kv}, hidden {hidden}, rank {rank}")
    cfg = oracle.ModelConfig(vocab=97, layers=2, dimensions=d, heads=heads, kv_heads=kv, hidden=hidden,
                             context=length + 4, dtype="bf16", **(dict(lora_rank=rank, lora_alpha=16.0) if rank else {}))
    weights = oracle.synthesize_weights(cfg, (45, 0), 0.05)
    for name in weights:
        if name.endswith("_adapter.up.weight"):
            weights[name] = oracle.bf16_encode(oracle.randn((46, len(name)), weights[name].size) * np.float32(0.1)).reshape(
                weights[name].shape)
    gpu = GpuLM(cfg, weights, kv_dtype)
    # The oracle that rounds its keys and values the same way.  A bf16 cache still rounds one that lies within the 2^-17 of the
    # projection from a boundary either way: 2^-8 of them, by 2^-8 each, 2^-12 of the keys and of the values of each of two
    # layers in the 2-norm, 2^-11 in all; twice that for the largest difference
    ref, allowed = oracle.OracleLM(cfg, weights, kv_bf16=kv_dtype == ct.BF16), 1e-4 if kv_dtype is None else 2.0**-10
    ids = oracle.random_ids((47, 0), batch * length, cfg.vocab).reshape(batch, length)
    rc, gc = ref.make_cache(batch), gpu.cache()
    for part in (ids, ids[:, :1], ids[:, :1]):  # the prompt, then steps over the keys and values that it stored
        assert rel_err(gpu.logits(part, gc), ref.logits(part, rc)[:, -1]) <= allowed


# rows, hidden, kernels of gate/up and down
SWIGLU = [(65, 1536, "mid, mid"), (128, 1536, "mid, mid"), (200, 1536, "mid, mid"), (513, 1536, "mid, mid"),
          (200, 1408, "mid, f32"), (3000, 1792, "tiles, mid")]


@pytest.mark.parametrize("rows,hidden,kernels", SWIGLU)
def test_swiglu_block_over_middling_rows(rows, hidden, kernels):
    say(f"case: SwiGLU module, {rows} rows, 512 -> {hidden} ({kernels})")
    rng = np.random.default_rng(rows)
    x = rng.standard_normal((rows, 512)).astype(np.float32)
    out = ct.C.c_void_p()
    ct.check(ct.lib().dl_swiglu_create(512, hidden, 0, ct.options(ct.BF16), ct.C.byref(out)))
    block = ct.Module(out)
    bits = {name: oracle.bf16_encode((0.05 * rng.standard_normal(t.shape)).astype(np.float32))
            for name, t in block.state().items()}
    block.load_state(bits, {name: ct.BF16 for name in bits})
    w = {name.split(".")[0]: oracle.bf16_decode(v).astype(np.float64) for name, v in bits.items()}
    gate, up = x @ w["gate"].T, x @ w["up"].T
    want = (gate / (1.0 + np.exp(-gate)) * up) @ w["down"].T
    got = block.forward(ct.Tensor.from_numpy(x, ct.F32, GPU)).numpy()
    agree(got, want, 2 * (bound(512) + bound(hidden)))  # both factors of a feature, then its sum
