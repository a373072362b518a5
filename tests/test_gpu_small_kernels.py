"""Sampling from logits that bound or break its f32 pre-selection, and RMSNorm over every width class, against the
oracle (sampling bit for bit)."""
import numpy as np
import pytest

import ctorch_amd as ct
import oracle
from common import say

pytestmark = pytest.mark.gpu
GPU = ct.device("gpu")


@pytest.mark.parametrize("vocab", [1, 3, 2048, 2049, 32000, 131072, 131073])
@pytest.mark.parametrize("temperature", [0.05, 0.8, 1.0, 40.0])
def test_sampling_is_bit_exact_whatever_the_logits_hold(vocab, temperature):
    say(f"case: dl_sample, vocab {vocab}, temperature {temperature}")
    rng = np.random.default_rng(vocab)
    rows = np.empty((9, vocab), np.float32)
    rows[:] = 3 * rng.standard_normal((9, vocab))
    rows[1] = 0.0                                               # the noise decides
    rows[2, rng.random(vocab) < 0.9] = -np.inf                  # masked entries
    rows[3] = -np.inf
    rows[4, vocab // 2] = np.inf
    rows[5, [vocab - 1, vocab // 3]] = np.nan
    rows[6] *= 1e37                                             # the scaled logits overflow f32
    rows[7] = np.float32(1e30) + np.zeros(vocab, np.float32)    # the noise is lost in the logits: ties
    rows[8] *= 1e-30
    for key in ((1, 2), (2**64 - 1, 77)):
        got = ct.sample(ct.Tensor.from_numpy(rows, ct.F32, GPU), temperature, key).numpy()
        assert np.array_equal(got, oracle.sample(rows, temperature, key)), key


def test_sampling_at_temperatures_beyond_f32():
    say("case: dl_sample at temperatures whose inverse f32 cannot hold")
    rows = np.random.default_rng(8).standard_normal((3, 5000)).astype(np.float32)
    for temperature in (1e-45, 1e-35, 1e35, 1e300):
        got = ct.sample(ct.Tensor.from_numpy(rows, ct.F32, GPU), temperature, (5, 6)).numpy()
        assert np.array_equal(got, oracle.sample(rows, temperature, (5, 6))), temperature


@pytest.mark.parametrize("width", [1, 4, 6, 1000, 1024, 1028, 2048, 4100, 8192, 8196])
@pytest.mark.parametrize("weight", [None, "f32", "bf16"])
def test_rms_norm_over_every_width_class(width, weight):
    say(f"case: rms_norm width {width}, weight {weight}")
    rng = np.random.default_rng(width)
    x, g = rng.standard_normal((5, width)).astype(np.float32), rng.uniform(0.5, 1.5, width).astype(np.float32)
    gw = None
    if weight == "f32":
        gw = ct.Tensor.from_numpy(g, ct.F32, GPU)
    elif weight == "bf16":
        bits = oracle.bf16_encode(g)
        g, gw = oracle.bf16_decode(bits), ct.Tensor.from_numpy(bits, ct.BF16, GPU)
    got = ct.rms_norm(ct.Tensor.from_numpy(x, ct.F32, GPU), [width], gw, 1e-5).numpy()
    want = x / np.sqrt(np.mean(x.astype(np.float64) ** 2, -1, keepdims=True) + 1e-5) * (1.0 if weight is None else g)
    # a thread's sum of at most width / 256 squares and ten more additions, halved by the root; four roundings after it
    assert np.all(np.abs(got - want) <= (4 + (width / 256 + 10) / 2) * 2.0**-23 * np.abs(want))
