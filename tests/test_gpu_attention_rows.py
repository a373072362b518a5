"""The general attention kernel (several positions, masks, head sizes 16 to 128) against numpy in 64 bits: edges of its
row tiles and key tiles, key splits, queries read through strides, and the causal chunks of a decoder against the oracle."""
import numpy as np
import pytest

import ctorch_amd as ct
import oracle
from common import build_pair, rel_err, say

pytestmark = pytest.mark.gpu
GPU = ct.device("gpu")


def reference(q, k, v, mask):
    group = q.shape[1] // k.shape[1]
    q, k, v = q.astype(np.float64), np.repeat(k, group, 1).astype(np.float64), np.repeat(v, group, 1).astype(np.float64)
    s = q @ k.transpose(0, 1, 3, 2) / np.sqrt(q.shape[-1])
    if mask is not None:
        s = np.where(mask, s, -np.inf)
    with np.errstate(invalid="ignore"):
        e = np.exp(s - s.max(-1, keepdims=True))
        return (e / e.sum(-1, keepdims=True)) @ v


@pytest.mark.parametrize("B,H,KV,L,S,D,bf16,masked", [
    (1, 2, 2, 1, 1, 16, False, False), (2, 3, 1, 5, 65, 32, False, True), (1, 8, 2, 4, 128, 64, True, False),
    (2, 12, 4, 11, 129, 64, False, True), (1, 4, 4, 65, 300, 128, True, True), (4, 32, 8, 7, 1508, 64, False, False),
    (1, 16, 2, 9, 700, 128, False, False), (1, 40, 2, 1, 200, 64, False, False), (2, 6, 2, 50, 50, 16, True, True)])
def test_attention_rows_match_64_bit_results(B, H, KV, L, S, D, bf16, masked):
    say(f"case: attention B={B} H={H} KV={KV} L={L} S={S} D={D} bf16={bf16} masked={masked}")
    rng = np.random.default_rng(S + L)
    q = rng.standard_normal((B, H, L, D)).astype(np.float32)
    k, v = (rng.standard_normal((B, KV, S, D)).astype(np.float32) for _ in range(2))
    if bf16:
        kb, vb = oracle.bf16_encode(k), oracle.bf16_encode(v)
        k, v = oracle.bf16_decode(kb), oracle.bf16_decode(vb)
        gk, gv = (ct.Tensor.from_numpy(a, ct.BF16, GPU) for a in (kb, vb))
    else:
        gk, gv = (ct.Tensor.from_numpy(a, ct.F32, GPU) for a in (k, v))
    masks = [None]
    if masked:
        shared = rng.random((B, 1, 1, S)) < 0.6
        shared[:, :, :, S // 2:] = False      # whole tiles dropped
        shared[:, :, :, 0] = True
        own = rng.random((1, H, L, S)) < 0.5
        own[0, 0, 0] = False                  # a row that keeps no key
        masks = [shared, own]
    want_nan = [m is not None and m.shape[1] > 1 for m in masks]
    for mask, nan in zip(masks, want_nan):
        gm = None if mask is None else ct.Tensor.from_numpy(mask, ct.BOOL, GPU)
        want = reference(q, k, v, mask)
        assert np.isnan(want).any() == nan
        got = ct.grouped_query_attention(ct.Tensor.from_numpy(q, ct.F32, GPU), gk, gv, gm).numpy()
        assert np.array_equal(np.isnan(got), np.isnan(want))
        # f32 sums: a score is off by some |score| 2^-24 sqrt(D), a weighted sum by 2^-24 sqrt(S)
        error = np.nan_to_num(got - want)
        assert np.linalg.norm(error) <= 2.0**-24 * (np.sqrt(D) + np.sqrt(S) + 8) * np.linalg.norm(np.nan_to_num(want))


# B, H, KV, L, S, D, kernel: 64 query rows to a work-group, a wave to each 16
MANY = [(4, 32, 8, 270, 275, D, "rows 4") for D in (16, 32, 64, 128)]


@pytest.mark.parametrize("bf16,masked", [(False, False), (False, True), (True, True)])
@pytest.mark.parametrize("B,H,KV,L,S,D,kernel", MANY)
def test_attention_over_many_rows_matches_64_bit_results(B, H, KV, L, S, D, kernel, bf16, masked):
    say(f"case: attention B={B} H={H} KV={KV} L={L} S={S} D={D} bf16={bf16} masked={masked} ({kernel})")
    rng = np.random.default_rng(D)
    q = rng.standard_normal((B, H, L, D)).astype(np.float32)
    k, v = (rng.standard_normal((B, KV, S, D)).astype(np.float32) for _ in range(2))
    encode = oracle.bf16_encode if bf16 else (lambda a: a)
    gk, gv = (ct.Tensor.from_numpy(encode(a), ct.BF16 if bf16 else ct.F32, GPU) for a in (k, v))
    if bf16:
        k, v = (oracle.bf16_decode(encode(a)) for a in (k, v))
    mask = None
    if masked:  # padding, and a row of its own per position that drops whole tiles of keys
        mask = (np.arange(S) < np.array([S, 200, 64, 1])[:, None])[:, None, None, :] & np.ones((B, 1, L, S), bool)
        mask[0, 0, 7, :] = False
        mask[0, 0, 7, 130] = True
    got = ct.grouped_query_attention(ct.Tensor.from_numpy(q, ct.F32, GPU), gk, gv,
                                     None if mask is None else ct.Tensor.from_numpy(mask, ct.BOOL, GPU)).numpy()
    want = reference(q, k, v, mask)
    bound = 2.0**-24 * (np.sqrt(D) + np.sqrt(S) + 8)
    assert np.linalg.norm(got - want) <= bound * np.linalg.norm(want)
    rows = np.linalg.norm(got - want, axis=-1) / np.linalg.norm(want, axis=-1)
    assert np.max(rows) <= 4 * bound


@pytest.mark.parametrize("L,S,masked", [(5, 130, False), (5, 130, True), (1, 70, True), (70, 90, False)])
@pytest.mark.parametrize("axis,start", [(0, 1), (1, 2), (2, 1), (3, 1)])
def test_views_of_a_query_and_a_mask_are_read_through_their_strides(L, S, masked, axis, start):
    say(f"case: attention, query narrowed along axis {axis} from {start}, L={L} S={S} masked={masked}")
    rng = np.random.default_rng(axis + S)
    shape = [2, 4, L, 32]
    view = lambda t, a, s, n: ct.Tensor(ct._new(ct.lib().dl_narrow, t.handle, a, s, n))
    stored = [n + (start + 1) * (i == axis) for i, n in enumerate(shape)]  # axis 3 from 1: rows off the 16-byte grid
    q = rng.standard_normal(stored).astype(np.float32)
    k, v = (rng.standard_normal((2, 2, S, 32)).astype(np.float32) for _ in range(2))
    gq = view(ct.Tensor.from_numpy(q, ct.F32, GPU), axis, start, shape[axis])
    gm = keep = None
    if masked:
        wide = rng.random((2, 1, L, S + 3)) < 0.6
        wide[..., 3] = True
        keep, gm = wide[..., 3:], view(ct.Tensor.from_numpy(wide, ct.BOOL, GPU), 3, 3, S)
    got = ct.grouped_query_attention(gq, *(ct.Tensor.from_numpy(a, ct.F32, GPU) for a in (k, v)), gm).numpy()
    q = np.take(q, range(start, start + shape[axis]), axis)
    want = reference(q, k, v, keep)
    assert np.linalg.norm(got - want) <= 2.0**-24 * (np.sqrt(32) + np.sqrt(S) + 8) * np.linalg.norm(want)


@pytest.mark.parametrize("bf16", [False, True])
def test_a_nan_value_under_the_mask_reaches_every_row_as_in_the_reference(bf16):
    say("case: attention, a NaN in V only under a mask that drops whole tiles")
    rng = np.random.default_rng(5)
    q, k, v = (rng.standard_normal(s).astype(np.float32) for s in ((1, 4, 3, 64), (1, 2, 256, 64), (1, 2, 256, 64)))
    mask = np.ones((1, 1, 1, 256), bool)
    mask[..., 128:] = False
    v[:, 0, 200, 3] = np.nan  # zero times NaN: head-dim entry 3 of the two query heads of KV head 0
    bits = (lambda a: ct.Tensor.from_numpy(oracle.bf16_encode(a), ct.BF16, GPU)) if bf16 else (
        lambda a: ct.Tensor.from_numpy(a, ct.F32, GPU))
    got = ct.grouped_query_attention(ct.Tensor.from_numpy(q, ct.F32, GPU), bits(k), bits(v),
                                     ct.Tensor.from_numpy(mask, ct.BOOL, GPU)).numpy()
    want = np.zeros(got.shape, bool)
    want[:, :2, :, 3] = True
    assert np.array_equal(np.isnan(got), want)


@pytest.mark.parametrize("batch,prefix,length,heads,kv,hd,kv_dtype", [
    (2, 100, 7, 8, 2, 64, None), (1, 700, 15, 8, 4, 128, None), (2, 63, 2, 8, 8, 64, ct.BF16), (3, 200, 33, 8, 2, 32, None),
    (1, 130, 20, 6, 2, 64, None)])
def test_causal_chunks_over_a_prefix_match_the_oracle(batch, prefix, length, heads, kv, hd, kv_dtype):
    say(f"case: {length} new positions over {prefix}, heads {heads}/{kv} of {hd}")
    cfg = oracle.ModelConfig(vocab=64, layers=2, dimensions=heads * hd, heads=heads, kv_heads=kv, hidden=256,
                             context=prefix + length + 2, dtype="f32")
    ref, gpu = build_pair(cfg, root=(91, 0), kv_dtype=kv_dtype)
    ids = oracle.random_ids((92, 0), batch * (prefix + length), cfg.vocab).reshape(batch, -1)
    rc, gc = ref.make_cache(batch), gpu.cache()
    bound = 1e-4 if kv_dtype is None else 2e-2
    for part in (ids[:, :prefix], ids[:, prefix:]):
        assert rel_err(gpu.logits(part, gc), ref.logits(part, rc)[:, -1]) <= bound


@pytest.mark.parametrize("batch,length", [(2, 0), (0, 3), (0, 20)])
@pytest.mark.parametrize("heads,kv,hd", [(8, 2, 32), (4, 2, 64), (4, 2, 8)])
def test_empty_queries_and_chunks_are_refused_and_leave_the_cache(batch, length, heads, kv, hd):
    say(f"case: empty attention, {batch} x {length}, heads {heads}/{kv} of {hd}")
    zeros = lambda *shape: ct.Tensor.from_numpy(np.zeros(shape, np.float32), ct.F32, GPU)
    q, k = zeros(batch, heads, length, hd), zeros(batch, kv, 70, hd)
    with pytest.raises(ct.DLError):
        ct.grouped_query_attention(q, k, k, None)
    empty = zeros(batch, length, heads * hd)
    decoder = ct.transformer_decoder(1, heads * hd, heads, kv, 64, 32, ct.F32, GPU, 10000.0)
    cache = ct.DecoderCache(decoder)
    with pytest.raises(ct.DLError):
        ct.decode(decoder, empty, cache)
    assert cache.length == 0
    if batch:  # the next chunk of that batch goes on as if the empty one had not been there
        assert ct.decode(decoder, zeros(batch, 3, heads * hd), cache).shape == (batch, 3, heads * hd)
        assert cache.length == 3
        with pytest.raises(ct.DLError):
            ct.decode(decoder, empty, cache)
        assert cache.length == 3


@pytest.mark.parametrize("D", [2, 4, 8])
@pytest.mark.parametrize("B,H,KV,L,S", [(2, 8, 2, 64, 65), (1, 4, 4, 5, 700), (2, 6, 3, 17, 130)])
def test_small_heads_with_and_without_key_splits(D, B, H, KV, L, S):
    say(f"case: attention B={B} H={H} KV={KV} L={L} S={S} D={D}")
    rng = np.random.default_rng(S + D)
    q = rng.standard_normal((B, H, L, D)).astype(np.float32)
    k, v = (rng.standard_normal((B, KV, S, D)).astype(np.float32) for _ in range(2))
    mask = rng.random((B, 1, L, S)) < 0.5
    mask[..., 0] = True
    for m in (None, mask):
        got = ct.grouped_query_attention(*(ct.Tensor.from_numpy(a, ct.F32, GPU) for a in (q, k, v)),
                                         None if m is None else ct.Tensor.from_numpy(m, ct.BOOL, GPU)).numpy()
        want = reference(q, k, v, m)
        assert np.linalg.norm(got - want) <= 2.0**-24 * (np.sqrt(D) + np.sqrt(S) + 8) * np.linalg.norm(want)
