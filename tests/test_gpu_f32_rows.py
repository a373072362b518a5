"""Projections with f32 weights over nine or more rows (the f32 matrix-core kernel), against numpy in 64 bits and the
CPU oracle: edges of its work-group shapes, partial weight tiles, K remainders, every epilogue."""
import numpy as np
import pytest

import ctorch_amd as ct
import oracle
from common import build_pair, rel_err, say

pytestmark = pytest.mark.gpu
GPU = ct.device("gpu")


# 16 k are summed in f32 and the sums of 16 in f64: at most 16 roundings of 2^-24 on each product, and one at the end
BOUND = 17 * 2.0**-24


@pytest.mark.parametrize("rows,k,n", [(9, 4, 1), (16, 36, 130), (17, 1000, 333), (33, 688, 64), (65, 32, 2),
                                      (129, 256, 8191), (700, 260, 2100), (2100, 64, 260)])
def test_linear_f32_weights_over_many_rows(rows, k, n):
    say(f"case: f32 linear {rows} x {k} -> {n}")
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
