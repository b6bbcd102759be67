"""The float (quantization-sensitive) BitLinear path and the packed STE backward on the GPU.

Against the oracle (double-accumulated restatement) and against the reference
build's own outputs (tests/golden/bitlinear_ref.npz): fp32 outputs within
1e-4 relative / 1e-5 absolute of the output scale (the north-star fp32 bound;
both sides sum in their own order), bf16 outputs within 2e-2 relative; the
normalised input of RMS_PERI is the bit-exact x * inv of the quantizer path."""
import os

import numpy as np
import pytest
import torch

from reimagined_amd import ops
from reimagined_amd._lib import call

pytestmark = pytest.mark.gpu
GOLDEN = os.path.join(os.path.dirname(__file__), "golden", "bitlinear_ref.npz")


def _close(got, want, rtol=1e-4, atol=1e-5, what=""):
    scale = max(float(np.abs(want).max()), 1e-30)
    np.testing.assert_allclose(got, want, rtol=rtol, atol=atol * scale, err_msg=what)


@pytest.mark.parametrize("m,k,n", [(40, 1024, 160), (40796 // 64, 1024, 160), (5, 1024, 160),
                                   (1, 1024, 160), (300, 1024, 8), (8192 // 8, 1024, 8),
                                   (1, 64, 3), (129, 256, 130), (17, 4096, 17), (16, 64, 16),
                                   (40796 // 16, 1024, 64), (100, 1000, 33), (33, 72, 48),
                                   (4097, 512, 64), (257, 1028, 17), (18, 4, 1)])
@pytest.mark.parametrize("rms", [False, True])
def test_linear_f32_matches_oracle(dev, orc, m, k, n, rms):
    rng = np.random.default_rng(m * 31 + n)
    x = (rng.standard_normal((m, k)) * rng.uniform(0.5, 4.0)).astype(np.float32)
    w = (rng.standard_normal((n, k)) / np.sqrt(k)).astype(np.float32)
    mag = rng.uniform(0.5, 1.5, n).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    t = lambda a: torch.from_numpy(a).to(dev)
    for mg, b in ((None, None), (mag, bias), (None, bias)):
        y = ops.linear_f32(t(x), t(w), rms, None if mg is None else t(mg),
                           None if b is None else t(b))
        want = orc.linear_f32(x, w, rms, mg, b)
        _close(y.cpu().numpy(), want, what=f"mag={mg is not None} bias={b is not None}")


@pytest.mark.parametrize("m,n,k", [(600, 160, 1024), (3, 160, 1024), (700, 8, 1024),
                                   (700, 64, 1024), (70, 40, 1028), (65, 33, 72)])
def test_linear_f32_bf16_io(dev, orc, m, n, k):
    rng = np.random.default_rng(m + n)
    x = rng.standard_normal((m, k)).astype(np.float32)
    w = (rng.standard_normal((n, k)) / np.sqrt(k)).astype(np.float32)
    xb = torch.from_numpy(x).to(torch.bfloat16)
    y = ops.linear_f32(xb.to(dev), torch.from_numpy(w).to(dev), True, out_dtype=torch.bfloat16)
    want = orc.linear_f32(xb.float().numpy(), w, True)
    _close(y.float().cpu().numpy(), want, rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("name", ["rms_mag_bias", "rms_mag", "exact", "exact_bias", "gate_rms_mag",
                                  "exact_wide_bias"])
def test_linear_f32_matches_reference_golden(dev, name):
    g = np.load(GOLDEN, allow_pickle=False)
    f = lambda key: (torch.from_numpy(g[f"{name}__{key}"].astype(np.float32)).to(dev)
                     if f"{name}__{key}" in g.files else None)
    exact = name.startswith("exact")
    y = ops.linear_f32(f("x"), f("w"), not exact, None if exact else f("mag"), f("bias"))
    _close(y.cpu().numpy(), g[f"{name}__y_float"], rtol=1e-5, atol=1e-6)


def _ste_case(orc, dev, x, w, grad, rms, mag, use_bias):
    o = orc.bitlinear_ste_backward(x, w, grad, rms, mag, use_bias)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    got = ops.bitlinear_ste_backward(t(x), t(o["q"]), t(o["act_scale"]), t(w),
                                     t(o["packed"].view(np.int32)), o["weight_scale"], t(grad),
                                     rms, None if mag is None else t(mag), use_bias)
    return o, {k: v.cpu().numpy() for k, v in got.items()}


@pytest.mark.parametrize("m,k,n", [(8, 256, 48), (300, 1024, 256), (1000, 512, 700),
                                   (33, 2048, 1024), (1, 16, 4), (257, 128, 132)])
@pytest.mark.parametrize("rms,with_mag,use_bias", [(True, True, True), (False, False, False),
                                                   (False, False, True), (True, True, False)])
def test_ste_backward_matches_oracle(dev, orc, m, k, n, rms, with_mag, use_bias):
    rng = np.random.default_rng(m + 7 * k + n)
    x = rng.standard_normal((m, k)).astype(np.float32)
    w = (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    grad = rng.standard_normal((m, n)).astype(np.float32)
    mag = rng.uniform(0.5, 1.5, n).astype(np.float32) if with_mag else None
    o, got = _ste_case(orc, dev, x, w, grad, rms, mag, use_bias)
    for key in ("dx", "dW", "dmag", "dbias"):
        if key in o:
            assert key in got
            _close(got[key], o[key], what=key)
    # the clip zeroes exactly the entries the oracle zeroes
    clip = np.abs(w / np.float32(o["weight_scale"] + np.float32(1e-8))) > 1.0
    assert np.all(got["dW"][clip] == 0.0)


@pytest.mark.parametrize("name", ["rms_mag_bias", "rms_mag", "exact", "exact_bias", "gate_rms_mag",
                                  "exact_wide_bias"])
def test_ste_backward_matches_reference_golden(dev, orc, name):
    g = np.load(GOLDEN, allow_pickle=False)
    f = lambda key: g[f"{name}__{key}"].astype(np.float32) if f"{name}__{key}" in g.files else None
    exact = name.startswith("exact")
    o, got = _ste_case(orc, dev, f("x"), f("w"), f("grad"), not exact, f("mag"),
                       f("bias") is not None)
    for key in ("dx", "dW", "dmag", "dbias"):
        if f"{name}__{key}" in g.files:
            _close(got[key], g[f"{name}__{key}"], rtol=1e-5, atol=1e-6, what=key)


@pytest.mark.parametrize("m,k,n", [(17, 4, 65), (63, 36, 66), (64, 64, 128), (65, 100, 129),
                                   (130, 1000, 72), (257, 1024, 160), (10300, 260, 33)])
@pytest.mark.parametrize("bf16,rms", [(False, False), (False, True), (True, False), (True, True)])
def test_linear_f32_error_bound(dev, m, k, n, bf16, rms):
    """The matrix products around their tiles' edges, rows and weights over twelve binades:
    within the rounding bound of a float sum of the row's products, K * 2^-24 of
    the sum of their magnitudes (and a few roundings of the norm and the affine)."""
    rng = np.random.default_rng(m + k + n)
    x = (rng.standard_normal((m, k)) * 2.0 ** rng.uniform(-6, 6, (m, k))).astype(np.float32)
    w = (rng.standard_normal((n, k)) * 2.0 ** rng.uniform(-6, 6, (n, k))).astype(np.float32)
    xt = torch.from_numpy(x).to(torch.bfloat16 if bf16 else torch.float32)
    y = ops.linear_f32(xt.to(dev), torch.from_numpy(w).to(dev), rms).cpu().numpy()
    xd = xt.double().numpy()
    if rms:
        xd = xd / np.sqrt((xd * xd).mean(1, keepdims=True) + 1e-6)
    want, size = xd @ w.astype(np.float64).T, np.abs(xd) @ np.abs(w.astype(np.float64)).T
    terms = k + 8 + (k if rms else 0)  # the RMS sum's own K roundings scale the row
    assert np.all(np.abs(y - want) <= terms * 2.0 ** -24 * size)


@pytest.mark.parametrize("bf16", [True, False])
def test_linear_f32_keeps_infinities(dev, bf16):
    """Infinities, NaN and values near the top of the range give what the float dot product
    gives: rows and columns that hold none are untouched."""
    rng = np.random.default_rng(3)
    m, k, n = 100, 96, 70
    x, w = (rng.standard_normal(s).astype(np.float32) for s in ((m, k), (n, k)))
    w = torch.from_numpy(w).to(torch.bfloat16).float().numpy()
    x[2, 3], x[5, 0], x[9, 95], x[40, 7] = np.inf, -np.inf, np.nan, 3.39e38
    w[6, 9], w[11, 2], w[12] = np.inf, np.nan, 1e-3
    xt = torch.from_numpy(x).to(torch.bfloat16 if bf16 else torch.float32)
    y = ops.linear_f32(xt.to(dev), torch.from_numpy(w).to(dev)).cpu().numpy()
    with np.errstate(invalid="ignore", over="ignore"):
        # the 3.39e38 row times its weights stays in range in float64 and past it in float32
        want = (xt.double().numpy()[:, None, :] * w.astype(np.float64)[None]).sum(-1).astype(np.float32)
    np.testing.assert_array_equal(np.isnan(y), np.isnan(want))
    np.testing.assert_array_equal(y[np.isinf(want)], want[np.isinf(want)])
    fine = np.isfinite(want)
    size = (np.abs(np.where(np.isfinite(x), x, 0)).astype(np.float64) @
            np.abs(np.where(np.isfinite(w), w, 0)).astype(np.float64).T)
    xs = xt.double().numpy()
    assert np.all(np.abs(y[fine] - want[fine]) <= ((k + 8) * 2.0 ** -24 * (size + 2.0 ** -6 * np.abs(want)))[fine])


@pytest.mark.parametrize("m,n", [(17, 64), (300, 100), (129, 128)])
@pytest.mark.parametrize("rms", [False, True])
def test_linear_f32_in_place(dev, m, n, rms):
    """y over x where a workgroup owns whole rows (M > 16, N = K <= 128): the same bits as y apart."""
    rng = np.random.default_rng(m + n)
    x, w = (torch.from_numpy(rng.standard_normal(s).astype(np.float32)).to(dev) for s in ((m, n), (n, n)))
    want = ops.linear_f32(x, w, rms)
    ws = torch.empty(m, device=dev)
    call("nsosx_linear_f32", x.data_ptr(), 0, m, n, w.data_ptr(), n, int(rms), None, None, x.data_ptr(), 0,
         ws.data_ptr(), None)
    torch.cuda.synchronize()
    assert torch.equal(x, want)
