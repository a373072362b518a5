"""RMSNorm over every width class, against 64-bit results."""
import numpy as np
import pytest

import ctorch_amd as ct
import oracle
from common import say

pytestmark = pytest.mark.gpu
GPU = ct.device("gpu")


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
