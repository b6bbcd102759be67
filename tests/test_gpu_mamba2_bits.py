"""The bits of the faithful Mamba-2 block and of its float projections.

The block quantizes the scan's output for its out_proj, so a last-bit change in the B / C / dt
projections or in the scan moves int8 codes, which is 2e-4 of the block's output: more than its
rounding, and what a saved activation or a resumed run would see.  The digests are those of the
float32 MFMA projections, of the lane chains of few rows and of the recurrence; a kernel that sums
in another order fails here.  Inputs come from numpy's generator alone.
"""
import hashlib

import numpy as np
import pytest
import torch

from reimagined_amd import layers, ops

pytestmark = pytest.mark.gpu

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
LINEAR = {  # m, k, n, input dtype, rms
    (700, 1024, 160, "f32", False): "5e9c1ab09fd58d33",
    (700, 1024, 160, "bf16", False): "0ee3e63dc3bbfa40",
    (257, 260, 65, "f32", True): "565bfa37f13b0e6b",
    (100, 768, 200, "bf16", True): "b20e9801210479c7",
    (10300, 264, 33, "f32", False): "db4f4f5ae48f67d9",
    (10300, 264, 64, "bf16", False): "2dbca9a6153b709c",
    (1500, 1024, 8, "f32", True): "2ea4bc44904a327a",
    (16, 1024, 160, "f32", False): "e1da4597b0e72f65",
    (5, 260, 70, "bf16", True): "9aeae8a526f57bde",
    (13, 2052, 160, "f32", False): "188e0f3307ab9f52",
    (9, 512, 2048, "bf16", False): "c34c21016c19cd3e",
}
BLOCK = {  # lengths, heads, d_state, dtype
    ((300, 1025), 16, 64, "f32"): "902fcd8100bd1db6",
    ((129, 40, 700), 8, 32, "f32"): "c8f260b96f539484",
    ((513, 64), 8, 64, "bf16"): "f3dd1b30973fa35b",
    ((257,), 8, 16, "f32"): "75ba4674e974701c",
}


def digest(*tensors):
    h = hashlib.sha256()
    for t in tensors:
        h.update(t.detach().cpu().contiguous().view(torch.uint8).numpy().tobytes())
    return h.hexdigest()[:16]


def linear(dev, m, k, n, dtype, rms):
    rng = np.random.default_rng(m + 3 * k + n)
    x, w = (torch.from_numpy(rng.standard_normal(s).astype(np.float32)) for s in ((m, k), (n, k)))
    return digest(ops.linear_f32(x.to(DTYPES[dtype]).to(dev), w.to(dev), rms))


def block(heads, d_state, dtype, seed):
    rng = np.random.default_rng(seed)
    d, inner = 32 * heads, 64 * heads
    n = lambda *s, std=1.0, mean=0.0: (rng.standard_normal(s) * std + mean).astype(np.float32)
    p = dict(w_x=n(inner, d, std=0.02), w_z=n(inner, d, std=0.02), w_B=n(d_state, d, std=d ** -0.5),
             w_C=n(d_state, d, std=d ** -0.5), w_dt=n(heads, d, std=d ** -0.5), w_out=n(d, inner, std=0.02),
             dt_bias=n(heads, std=0.5, mean=-2.0), conv_w=n(inner + 2 * d_state, 4, std=0.5),
             conv_b=n(inner + 2 * d_state, std=0.1), a_log=n(heads), d_skip=n(heads),
             norm_w=n(inner, std=0.1, mean=1.0), H=heads, P=64, N=d_state, G=1)
    return layers.Mamba2Block(p, dtype=DTYPES[dtype]), n, d


def prefill(dev, lengths, heads, d_state, dtype):
    layer, n, d = block(heads, d_state, dtype, sum(lengths) + d_state)
    u = torch.from_numpy(n(sum(lengths), d)).to(DTYPES[dtype]).to(dev)
    cu = torch.from_numpy(np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)).to(dev)
    r = layer.forward(u, cu)
    return digest(r["out"], r["final_state"])


@pytest.mark.parametrize("case", LINEAR)
def test_linear_bits(dev, case):
    assert linear(dev, *case) == LINEAR[case]


@pytest.mark.parametrize("case", BLOCK)
def test_block_prefill_bits(dev, case):
    assert prefill(dev, list(case[0]), *case[1:]) == BLOCK[case]
