"""A decoder layer over so many rows that its projections take the largest work-groups of their kernels (gemm_tiles with
partial column blocks and LoRA, gemm_f32's 64 x 64 and 128 x 128), every position against numpy in 64 bits.
test_host_rules.py checks on the CPU that each projection takes the kernel named here."""
import numpy as np
import pytest

import ctorch_amd as ct
import oracle
from common import agree, say

pytestmark = pytest.mark.gpu
GPU = ct.device("gpu")
ALPHA = 32.0

# batch, length, d, heads, kv, hidden, rank, dtype, kernels of QKV, output, gate/up and down, error bound.  Split
# activations leave 2^-17 in each of three projections; f32 ones sums of 16 roundings of 2^-24, and the attention 16 more
# (its heads are 32 wide there: at 64 and 128 the prefill kernel splits queries, keys and values into two bf16 parts, 2^-17)
LAYERS = [(128, 129, 512, 8, 1, 320, 16, "bf16", "tiles, tiles, tiles, tiles", 3 * 2.0**-17),
          (130, 127, 512, 8, 1, 320, 0, "bf16", "tiles, tiles, tiles, tiles", 3 * 2.0**-17),
          (64, 130, 256, 8, 2, 256, 8, "f32", "f32 64x64, f32 64x64, f32 64x64, f32 64x64", 32 * 2.0**-24),
          (256, 128, 512, 16, 16, 256, 0, "f32", "f32 128x128, f32 128x128, f32 128x128, f32 128x128", 32 * 2.0**-24)]


def rms(x, w):
    return x / np.sqrt(np.mean(x * x, -1, keepdims=True) + 1e-5) * w


def layer_reference(x, w, heads, kv, rank):
    """One layer and the final norm in 64 bits (w: the decoder's state without "layer0.")."""
    b, n, d = x.shape
    hd = d // heads

    def rotate(t):
        c, s = w["attention.rotary.cosine"][:n], w["attention.rotary.sine"][:n]
        even, odd = t[..., 0::2], t[..., 1::2]
        return np.stack([even * c - odd * s, even * s + odd * c], -1).reshape(t.shape)

    h = rms(x, w["attention_norm.weight"]).reshape(-1, d)
    q, k, v = (h @ w[f"attention.{name}.weight"].T for name in ("query", "key", "value"))
    if rank:
        for out, name in ((q, "query"), (v, "value")):
            out += ALPHA / rank * (h @ w[f"attention.{name}_adapter.down.weight"].T) @ w[f"attention.{name}_adapter.up.weight"].T
    q, k, v = (t.reshape(b, n, -1, hd).transpose(0, 2, 1, 3) for t in (q, k, v))
    q, k = rotate(q), rotate(k)
    late = np.triu(np.ones((n, n), bool), 1)
    out = np.empty((b, n, heads, hd))
    for i in range(heads):
        s = q[:, i] @ k[:, i * kv // heads].transpose(0, 2, 1) / np.sqrt(hd)
        s[:, late] = -np.inf
        e = np.exp(s - s.max(-1, keepdims=True))
        out[:, :, i] = (e / e.sum(-1, keepdims=True)) @ v[:, i * kv // heads]
    x = x + (out.reshape(-1, d) @ w["attention.output.weight"].T).reshape(x.shape)
    h = rms(x, w["feedforward_norm.weight"]).reshape(-1, d)
    gate, up = h @ w["feedforward.gate.weight"].T, h @ w["feedforward.up.weight"].T
    x = x + ((gate / (1.0 + np.exp(-gate)) * up) @ w["feedforward.down.weight"].T).reshape(x.shape)
    return rms(x, w["normalization.weight"])


@pytest.mark.parametrize("batch,length,d,heads,kv,hidden,rank,dtype,kernels,bound", LAYERS)
def test_a_layer_over_many_rows_matches_64_bit_results(batch, length, d, heads, kv, hidden, rank, dtype, kernels, bound):
    say(f"case: {dtype} layer over {batch} x {length} positions, d {d}, heads {heads}/{kv}, hidden {hidden}, rank {rank}")
    kind = ct.BF16 if dtype == "bf16" else ct.F32
    decoder = ct.transformer_decoder(1, d, heads, kv, hidden, length, kind, GPU)
    if rank:
        ct.check(ct.lib().dl_transformer_decoder_attach_lora(decoder.handle, rank, ALPHA, 1, 1))
    rng = np.random.default_rng(d + rank)
    state, w = decoder.state(), {}
    for name in sorted(state):
        short = name.removeprefix("layer0.")
        if ".rotary." in name:
            w[short] = state[name].numpy().astype(np.float64)
            continue
        value = (rng.uniform(0.8, 1.2, state[name].shape) if name.endswith("norm.weight") or name == "normalization.weight"
                 else rng.standard_normal(state[name].shape) * (0.2 if "adapter.up" in name else 1.0) / np.sqrt(d))
        value = value.astype(np.float32)
        stored = oracle.bf16_encode(value) if dtype == "bf16" else value
        w[short] = (oracle.bf16_decode(stored) if dtype == "bf16" else value).astype(np.float64).reshape(state[name].shape)
        state[name] = ct.Tensor.from_numpy(stored.reshape(state[name].shape), kind, GPU)
    decoder.load_state(state)
    x = rng.standard_normal((batch, length, d)).astype(np.float32)
    got = ct.decode(decoder, ct.Tensor.from_numpy(x, ct.F32, GPU), ct.DecoderCache(decoder)).numpy()
    want = layer_reference(x.astype(np.float64), w, heads, kv, rank)
    agree(got.reshape(-1, d), want.reshape(-1, d), bound)
