"""The work that a user has this library do, as measurable cases: token generation, decoder steps and prefills through
the decoder's own entry, and the operators that programs call beside it.

A case is a dict of plain values with a "kind":

  generate   DecoderLM.generate: a prompt through the model, then greedy tokens (the serving loop; a whole call)
  decode     TransformerDecoder.decode of `length` new positions of `batch` sequences over `prefix` cached ones: one
             position is a step of a caller's own token loop, a few are the verification of drafted tokens, many are
             the prefill of a prompt (or of one chunk of it)
  linear     ct.linear over `rows` rows (the LM head over every position of a text, a projection of its own)
  swiglu     the SwiGLU block as a module of its own
  attention  ct.grouped_query_attention without a causal window, with or without a padding mask
  sample     ct.sample of a batch of logits

Weights and inputs are drawn from the seed in device memory.  Outputs are zero-copy views of the library's tensors.
"""
import ctypes
import math

import numpy as np
import torch

import ctorch_amd as ct

# The widths that the tests and the benchmark use: the tiny f32 byte model, the 1B and the 8B decoder (bf16 weights).
MODELS = {
    "tiny": dict(vocab=256, layers=4, d=256, heads=8, kv=2, hidden=688, base=10000.0, dtype="f32"),
    "1b": dict(vocab=32000, layers=16, d=2048, heads=32, kv=8, hidden=5632, base=10000.0, dtype="bf16"),
    "8b": dict(vocab=32000, layers=32, d=4096, heads=32, kv=8, hidden=14336, base=500000.0, dtype="bf16"),
}
DTYPE = {"f32": ct.F32, "bf16": ct.BF16}
NORM_EPSILON = 1e-5
LORA_ALPHA = 32.0


def listed():
    return [
        # the smallest model end to end: a 32-byte prompt and 128 bytes of text (launches and latency count)
        dict(name="generate_tiny", kind="generate", model="tiny", batch=1, prefix=0, prompt=32, steps=128, cache="f32"),
        # one chat request to the 1B model: a 128-token prompt, 32 tokens of answer, the default f32 cache
        dict(name="generate_1b", kind="generate", model="1b", batch=1, prefix=0, prompt=128, steps=32, cache="f32"),
        # a serving batch in flight: 32 sequences of 2048 cached tokens each, bf16 cache, 16 more tokens
        dict(name="generate_1b_batch", kind="generate", model="1b", batch=32, prefix=2048, prompt=1, steps=16,
             cache="bf16"),
        # long-context decode at 8B widths: one position of 8 sequences over 32768 cached ones
        dict(name="decode_8b_long", kind="decode", model="8b", layers=2, batch=8, prefix=32768, length=1, cache="bf16",
             lora=0),
        # drafted tokens verified: 7 new positions of 4 sequences of a ragged length
        dict(name="verify_1b", kind="decode", model="1b", layers=4, batch=4, prefix=1501, length=7, cache="f32", lora=0),
        # an ordinary prompt, shorter than a full tile of rows
        dict(name="prompt_1b", kind="decode", model="1b", layers=4, batch=1, prefix=0, length=200, cache="f32", lora=0),
        # a prompt of odd length at 8B widths into the bf16 cache
        dict(name="prompt_8b", kind="decode", model="8b", layers=2, batch=1, prefix=0, length=1013, cache="bf16", lora=0),
        # the largest: a batch of long prompts with unmerged LoRA adapters
        dict(name="prefill_1b_lora", kind="decode", model="1b", layers=2, batch=4, prefix=0, length=4096, cache="f32",
             lora=16),
        # f32 weights, the library's default dtype: a batch of byte texts through the tiny model
        dict(name="prompt_tiny", kind="decode", model="tiny", layers=4, batch=4, prefix=0, length=510, cache="f32",
             lora=0),
        # a text scored: the LM head over each of its positions
        dict(name="head_1b", kind="linear", rows=333, inputs=2048, outputs=32000, dtype="bf16", bias=False),
        # bidirectional attention over a padded batch
        dict(name="attention_padded", kind="attention", batch=4, heads=32, kv=8, length=500, source=500, head_dim=64,
             dtype="f32", mask=True),
        # the next token of 32 sequences drawn from logits the caller holds
        dict(name="sample_1b", kind="sample", rows=32, vocab=32000, temperature=0.8),
    ]


def _log(rng, low, high):
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    kind = rng.choice(["generate", "decode", "decode", "verify", "prefill", "prefill", "prefill", "linear", "swiglu",
                       "attention", "sample"])
    cache = rng.choice(["f32", "bf16"])
    if kind == "generate":
        model = rng.choice(["tiny", "1b"])
        batch = _log(rng, 1, 32)
        return dict(kind="generate", model=model, batch=batch, prefix=0,
                    prompt=_log(rng, 1, 400 if batch <= 4 else 64), steps=_log(rng, 4, 100 if model == "tiny" else 24),
                    cache=cache)
    if kind == "decode":
        batch = _log(rng, 1, 64)
        return dict(kind="decode", model=rng.choice(["1b", "8b"]), layers=2, batch=batch,
                    prefix=_log(rng, 16, 200000 // batch if batch > 6 else 30000), length=1, cache=cache,
                    lora=rng.choice([0, 0, 16]))
    if kind == "verify":
        return dict(kind="decode", model=rng.choice(["1b", "8b"]), layers=2, batch=_log(rng, 1, 8),
                    prefix=_log(rng, 16, 6000), length=rng.randint(2, 15), cache=cache, lora=0)
    if kind == "prefill":
        model = rng.choice(["tiny", "1b", "1b", "8b"])
        batch = _log(rng, 1, 8)
        return dict(kind="decode", model=model, layers=2, batch=batch,
                    prefix=rng.choice([0, 0, _log(rng, 16, 1024)]), length=_log(rng, 16, 4096 // batch), cache=cache,
                    lora=rng.choice([0, 0, 16]))
    if kind == "linear":
        dtype = rng.choice(["bf16", "bf16", "f32"])
        return dict(kind="linear", rows=_log(rng, 1, 2000), inputs=rng.choice([512, 1000, 2048, 4096]),
                    outputs=_log(rng, 250, 16000), dtype=dtype, bias=rng.choice([True, False]))
    if kind == "swiglu":
        model = rng.choice(["tiny", "1b", "8b"])
        return dict(kind="swiglu", model=model, rows=_log(rng, 1, 2000))
    if kind == "attention":
        length = _log(rng, 2, 700)
        return dict(kind="attention", batch=rng.randint(1, 4), heads=rng.choice([8, 16, 32]), kv=rng.choice([2, 4, 8]),
                    length=length, source=length + rng.choice([0, rng.randint(1, 300)]),
                    head_dim=rng.choice([32, 64, 128]), dtype=rng.choice(["f32", "bf16"]), mask=rng.random() < 0.6)
    return dict(kind="sample", rows=_log(rng, 1, 64), vocab=_log(rng, 200, 130000),
                temperature=rng.choice([0.0, 0.7, 1.0]))


# ------------------------------------------------------------------------------------------------ inputs
class _View:
    """A library tensor as a device array (the view holds the tensor)."""

    _TYPES = {ct.F32: ("<f4", 4), ct.I64: ("<i8", 8), ct.BF16: ("<i2", 2)}

    def __init__(self, tensor):
        lib = ct.lib()
        kind, size = self._TYPES[tensor.dtype]
        shape = tensor.shape
        strides = lib.dl_tensor_strides(tensor.handle)
        self.tensor = tensor
        self.__cuda_array_interface__ = dict(
            shape=shape, typestr=kind, version=3, data=(lib.dl_tensor_data(tensor.handle), False),
            strides=tuple(strides.data[i] * size for i in range(len(shape))))


def _torch(tensor):
    view = torch.as_tensor(_View(tensor), device="cuda")
    return view.view(torch.bfloat16) if tensor.dtype == ct.BF16 else view


def _normal(key, slot, shape, scale, dtype="f32"):
    return ct.normal(ct.fold_in(key, slot), list(shape), scale, DTYPE[dtype])


def _host(array, dtype="f32"):
    if dtype == "bf16":
        bits = torch.from_numpy(np.asarray(array, np.float32)).to(torch.bfloat16).view(torch.int16).numpy()
        return ct.Tensor.from_numpy(bits.view(np.uint16), ct.BF16, ct.device("gpu"))
    return ct.Tensor.from_numpy(np.asarray(array, np.float32), ct.F32, ct.device("gpu"))


def _decoder(case, key, context):
    """A decoder with N(0, 0.02) projections, norm weights around 1, and adapters that matter where it has them."""
    m = MODELS[case["model"]]
    layers = case.get("layers", m["layers"])
    decoder = ct.transformer_decoder(layers, m["d"], m["heads"], m["kv"], m["hidden"], context, DTYPE[m["dtype"]],
                                     ct.device("gpu"), m["base"], kv_dtype=DTYPE[case["cache"]])
    if case.get("lora"):
        ct.check(ct.lib().dl_transformer_decoder_attach_lora(decoder.handle, case["lora"], LORA_ALPHA, 1, 1))
    rng = np.random.default_rng(key[0])
    state = decoder.state()
    for slot, name in enumerate(sorted(state)):
        if ".rotary." in name:
            continue
        if name.endswith("norm.weight") or name == "normalization.weight":
            state[name] = _host(rng.uniform(0.8, 1.2, state[name].shape), m["dtype"])
        else:
            state[name] = _normal(key, slot, state[name].shape, 0.02, m["dtype"])
    decoder.load_state(state)
    return decoder


def _cache(case, decoder, key):
    """A cache that holds `prefix` positions of N(0, 1) keys and values."""
    m = MODELS[case["model"]]
    cache = ct.DecoderCache(decoder)
    if case["prefix"]:
        shape = [case["batch"], m["kv"], case["prefix"], m["d"] // m["heads"]]
        for layer in range(case.get("layers", m["layers"])):
            cache.append(layer, _normal(key, 5000 + 2 * layer, shape, 1.0, case["cache"]),
                         _normal(key, 5001 + 2 * layer, shape, 1.0, case["cache"]))
    return cache


def prepare(case, seed):
    key = (int(seed) + 1, 77)
    rng = np.random.default_rng([int(seed), 3])
    kind = case["kind"]
    if kind == "generate":
        m = MODELS[case["model"]]
        decoder = _decoder(case, key, case["prefix"] + case["prompt"] + case["steps"] + 8)
        # The head's rows are the embedding's in another order, so that each step prefers one token clearly, as a
        # trained model mostly does, and no rounding decides the text.
        embedding = _normal(key, 9000, (m["vocab"], m["d"]), 1.0, m["dtype"])
        order = ct.Tensor.from_numpy(rng.permutation(m["vocab"]).astype(np.int64), ct.I64, ct.device("gpu"))
        head = ct.embedding(order, embedding)
        state = dict(kind=kind, decoder=decoder, embedding=embedding, head=head, steps=case["steps"],
                     prefix=case["prefix"], cache=_cache(case, decoder, key),
                     ids=rng.integers(0, m["vocab"], (case["batch"], case["prompt"]), dtype=np.int64))
        state["lm"] = ct.DecoderLM(ct.embedding_from(embedding), decoder, ct.linear_from(head))
    elif kind == "decode":
        m = MODELS[case["model"]]
        decoder = _decoder(case, key, case["prefix"] + case["length"] + 8)
        state = dict(kind=kind, decoder=decoder, cache=_cache(case, decoder, key), prefix=case["prefix"],
                     x=_normal(key, 9001, (case["batch"], case["length"], m["d"]), 1.0))
    elif kind == "linear":
        state = dict(kind=kind, x=_normal(key, 1, (case["rows"], case["inputs"]), 1.0),
                     w=_normal(key, 2, (case["outputs"], case["inputs"]), 0.02, case["dtype"]),
                     b=_normal(key, 3, (case["outputs"],), 0.1, case["dtype"]) if case["bias"] else None)
    elif kind == "swiglu":
        m = MODELS[case["model"]]
        out = ctypes.c_void_p()
        ct.check(ct.lib().dl_swiglu_create(m["d"], m["hidden"], 0, ct.options(DTYPE[m["dtype"]]), ctypes.byref(out)))
        block = ct.Module(out)
        weights = {name: _normal(key, slot, t.shape, 0.02, m["dtype"])
                   for slot, (name, t) in enumerate(sorted(block.state().items()))}
        block.load_state(weights)
        state = dict(kind=kind, block=block, x=_normal(key, 100, (case["rows"], m["d"]), 1.0))
    elif kind == "attention":
        b, d = case["batch"], case["head_dim"]
        mask = None
        if case["mask"]:  # each sequence keeps its own number of keys, from the front
            kept = rng.integers(max(1, case["source"] // 3), case["source"] + 1, b)
            mask = ct.Tensor.from_numpy((np.arange(case["source"])[None, :] < kept[:, None])[:, None, None, :], ct.BOOL,
                                        ct.device("gpu"))
        state = dict(kind=kind, mask=mask, q=_normal(key, 1, (b, case["heads"], case["length"], d), 1.0),
                     k=_normal(key, 2, (b, case["kv"], case["source"], d), 1.0, case["dtype"]),
                     v=_normal(key, 3, (b, case["kv"], case["source"], d), 1.0, case["dtype"]))
    else:
        state = dict(kind=kind, logits=_normal(key, 1, (case["rows"], case["vocab"]), 3.0),
                     temperature=case["temperature"], key=ct.fold_in(key, 2))
    ct.synchronize()
    return state


def run(state):
    kind = state["kind"]
    if kind == "generate":
        state["cache"].truncate(state["prefix"])
        tokens, last = state["lm"].generate(state["ids"], state["cache"], state["steps"], host=False)
        return {"tokens": _torch(tokens), "logits": _torch(last)}
    if kind == "decode":
        state["cache"].truncate(state["prefix"])
        return _torch(ct.decode(state["decoder"], state["x"], state["cache"]))
    if kind == "linear":
        return _torch(ct.linear(state["x"], state["w"], state["b"]))
    if kind == "swiglu":
        return _torch(state["block"].forward(state["x"]))
    if kind == "attention":
        return _torch(ct.grouped_query_attention(state["q"], state["k"], state["v"], state["mask"]))
    return _torch(ct.sample(state["logits"], state["temperature"], state["key"]))


# ------------------------------------------------------------------------------------------------ accounts
def _chunk_work(case, m, layers, batch, prefix, length, first=True):
    """Bytes and operations of one decoder chunk: weights once, cached keys and values read once, new ones written."""
    e = 4 if m["dtype"] == "f32" else 2
    c = 4 if case["cache"] == "f32" else 2
    d, hd = m["d"], m["d"] // m["heads"]
    kv = m["kv"] * hd
    r = case.get("lora", 0)
    weights = d * d * 2 + 2 * kv * d + 3 * m["hidden"] * d + r * (3 * d + kv)
    pairs = length * prefix + length * (length + 1) // 2
    rows = batch * length
    return {"bytes": layers * (weights * e + 2 * batch * kv * (prefix + length) * c) + rows * d * 8,
            "flops": layers * (2 * weights * rows + 4 * batch * pairs * m["heads"] * hd)}


def work(case):
    kind = case["kind"]
    if kind == "generate":
        m = MODELS[case["model"]]
        e = 4 if m["dtype"] == "f32" else 2
        head = m["vocab"] * m["d"]
        chunks = [case["prompt"]] + [1] * (case["steps"] - 1)
        total = {"bytes": 0, "flops": 0}
        at = case["prefix"]
        for n in chunks:
            w = _chunk_work(case, m, m["layers"], case["batch"], at, n)
            total["bytes"] += w["bytes"] + head * e + case["batch"] * m["vocab"] * 4
            total["flops"] += w["flops"] + 2 * head * case["batch"]
            at += n
        return total
    if kind == "decode":
        m = MODELS[case["model"]]
        return _chunk_work(case, m, case["layers"], case["batch"], case["prefix"], case["length"])
    if kind == "linear":
        e = 4 if case["dtype"] == "f32" else 2
        r, k, n = case["rows"], case["inputs"], case["outputs"]
        return {"bytes": n * k * e + (n * e if case["bias"] else 0) + 4 * r * (k + n), "flops": 2 * r * k * n}
    if kind == "swiglu":
        m = MODELS[case["model"]]
        e = 4 if m["dtype"] == "f32" else 2
        return {"bytes": 3 * m["d"] * m["hidden"] * e + 8 * case["rows"] * m["d"],
                "flops": 6 * case["rows"] * m["d"] * m["hidden"]}
    if kind == "attention":
        e = 4 if case["dtype"] == "f32" else 2
        b, s, d = case["batch"], case["source"], case["head_dim"]
        queries = b * case["heads"] * case["length"]
        return {"bytes": 8 * queries * d + 2 * e * b * case["kv"] * s * d, "flops": 4 * queries * s * d}
    return {"bytes": case["rows"] * (case["vocab"] * 4 + 8), "flops": 0}


def tolerance(case):
    """About four times what results differ from 64-bit ones by.  bf16 weights meet activations that are split into two
    bf16 parts (2^-17 each: 2.5e-6 to 6e-6 measured for a layer, 1e-5 for the 16-layer model); f32 weights and the
    attention operator are f32 sums (1e-7 to 5e-7).  A bf16 cache rounds each new key and value, and one near a
    rounding boundary may go either way (1.6e-4 over a prompt of which every key is new)."""
    kind = case["kind"]
    if kind == "sample":
        return "exact"
    if kind == "attention":
        return {"rel": 4e-6, "max": 1e-3}
    if kind == "linear" or kind == "swiglu":
        f32 = (case if kind == "linear" else MODELS[case["model"]])["dtype"] == "f32"
        return {"rel": 4e-6 if f32 else 2e-5, "max": 1e-3}
    return {"rel": 6e-4 if case["cache"] == "bf16" else 4e-5, "max": 2e-2, "differ": 0.0}


# ------------------------------------------------------------------------------------------------ 64-bit results
def _exact_tensor(tensor):
    """A library tensor's values on the host, in 64 bits."""
    array = tensor.numpy()
    if tensor.dtype == ct.BF16:
        return torch.from_numpy(array.view(np.int16)).view(torch.bfloat16).double()
    return torch.from_numpy(array).double()


def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + NORM_EPSILON) * w


def _rotate(x, cosine, sine):
    even, odd = x[..., 0::2], x[..., 1::2]
    return torch.stack([even * cosine - odd * sine, even * sine + odd * cosine], -1).flatten(-2)


def _attend(q, k, v, first):
    """Causal grouped-query attention of q [b, h, n, e] over k, v [b, g, first + n, e], a block of rows at a time."""
    b, h, n, e = q.shape
    g = k.shape[1]
    out = torch.empty_like(q)
    for l in range(0, n, 1024):
        rows = min(1024, n - l)
        seen = first + l + rows
        late = torch.arange(seen)[None, :] > first + l + torch.arange(rows)[:, None]
        for j in range(b):
            for i in range(g):
                heads = slice(i * h // g, (i + 1) * h // g)
                p = torch.matmul(q[j, heads, l:l + rows].reshape(-1, e), k[j, i, :seen].T).mul_(1.0 / math.sqrt(e))
                p = p.view(-1, rows, seen).masked_fill_(late, -math.inf)
                out[j, heads, l:l + rows] = torch.matmul(torch.softmax(p, -1), v[j, i, :seen])
    return out


class _Exact:
    """The decoder in plain 64-bit torch on the host.  The rotation tables are the module's (f32 buffers of its
    state), and keys and values are rounded to the cache's type, as both are part of what the caller chose."""

    def __init__(self, case, state):
        self.m = MODELS[case["model"]]
        self.layers = case.get("layers", self.m["layers"])
        self.round = case["cache"] == "bf16"
        self.scale = LORA_ALPHA / case["lora"] if case.get("lora") else 0.0
        tensors = state["decoder"].state()
        rotary = "layer0.attention.rotary."
        self.cosine, self.sine = _exact_tensor(tensors[rotary + "cosine"]), _exact_tensor(tensors[rotary + "sine"])
        self.w = {name: _exact_tensor(t) for name, t in tensors.items() if ".rotary." not in name}
        self.room = state["prefix"] + case.get("length", 0) + case.get("prompt", 0) + case.get("steps", 0)
        self.at = [0] * self.layers
        self.k, self.v = ([torch.empty(case["batch"], self.m["kv"], self.room, self.m["d"] // self.m["heads"],
                                       dtype=torch.float64) for _ in range(self.layers)] for _ in range(2))
        if state["prefix"]:
            held = state["cache"].state()
            for i in range(self.layers):
                self.append(i, _exact_tensor(held["past_key_%d" % i]), _exact_tensor(held["past_value_%d" % i]))

    def append(self, i, k, v):
        to = slice(self.at[i], self.at[i] + k.shape[2])
        for held, new in ((self.k[i], k), (self.v[i], v)):
            held[:, :, to] = new.to(torch.bfloat16).double() if self.round else new
        self.at[i] = to.stop

    def chunk(self, x):
        m, w = self.m, self.w
        b, n, d = x.shape
        for i in range(self.layers):
            a, f = "layer%d.attention." % i, "layer%d.feedforward." % i
            h = _rms(x, w["layer%d.attention_norm.weight" % i])
            q, k, v = (h @ w[a + name + ".weight"].T for name in ("query", "key", "value"))
            if self.scale:
                q += self.scale * (h @ w[a + "query_adapter.down.weight"].T) @ w[a + "query_adapter.up.weight"].T
                v += self.scale * (h @ w[a + "value_adapter.down.weight"].T) @ w[a + "value_adapter.up.weight"].T
            q, k, v = (t.view(b, n, -1, d // m["heads"]).transpose(1, 2) for t in (q, k, v))
            first = self.at[i]
            c, s = self.cosine[first:first + n], self.sine[first:first + n]
            self.append(i, _rotate(k, c, s), v)
            seen = self.at[i]
            out = _attend(_rotate(q, c, s), self.k[i][:, :, :seen], self.v[i][:, :, :seen], first)
            x = x + out.transpose(1, 2).reshape(b, n, d) @ w[a + "output.weight"].T
            h = _rms(x, w["layer%d.feedforward_norm.weight" % i])
            h = torch.nn.functional.silu(h @ w[f + "gate.weight"].T) * (h @ w[f + "up.weight"].T)
            x = x + h @ w[f + "down.weight"].T
        return _rms(x, w["normalization.weight"])


def exact(case, seed):
    state = prepare(case, seed)
    kind = case["kind"]
    if kind == "generate":
        model = _Exact(case, state)
        embedding, head = _exact_tensor(state["embedding"]), _exact_tensor(state["head"])
        ids, tokens = torch.from_numpy(state["ids"]), []
        for _ in range(case["steps"]):
            logits = model.chunk(embedding[ids])[:, -1] @ head.T
            ids = logits.argmax(-1, keepdim=True)
            tokens.append(ids)
        return {"tokens": torch.cat(tokens, 1), "logits": logits}
    if kind == "decode":
        return _Exact(case, state).chunk(_exact_tensor(state["x"]))
    if kind == "linear":
        y = _exact_tensor(state["x"]) @ _exact_tensor(state["w"]).T
        return y + _exact_tensor(state["b"]) if case["bias"] else y
    if kind == "swiglu":
        w = {name.split(".")[0]: _exact_tensor(t) for name, t in state["block"].state().items()}
        x = _exact_tensor(state["x"])
        return (torch.nn.functional.silu(x @ w["gate"].T) * (x @ w["up"].T)) @ w["down"].T
    if kind == "attention":
        q, k, v = (_exact_tensor(state[n]) for n in "qkv")
        k, v = (t.repeat_interleave(case["heads"] // case["kv"], 1) for t in (k, v))
        s = q @ k.transpose(2, 3) / math.sqrt(case["head_dim"])
        if case["mask"]:
            s.masked_fill_(~torch.from_numpy(state["mask"].numpy()), -math.inf)
        return s.softmax(-1) @ v
    return None
