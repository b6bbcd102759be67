"""The straight-through backward's split contractions against float64 on the same codes, at the
edges of their tiles (128 x 256 outputs, 32-deep stages) and with gradients that are not finite.

Each bf16 piece's product with a code is exact, so only the float sums round: n products added
in any order stay within n * 2^-24 of the sum of their magnitudes (plus the last scaling's two
roundings and the gradient's own, 4 * 2^-24)."""
import numpy as np
import pytest
import torch

from reimagined_amd import ops
from reimagined_amd._lib import call, lib

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


def _case(dev, m, k, n, with_mag, seed, spread=1.0):
    rng = np.random.default_rng(seed)
    w = (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    packed, ws = ops.pack_ternary(w)
    codes = ops.unpack_ternary(packed, n * k).reshape(n, k).astype(np.float64)
    x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).to(dev)
    q, s = ops.quantize_activations_bitnet(x, 8)
    grad = (rng.standard_normal((m, n)) * spread ** rng.uniform(-1, 1, (m, n))).astype(np.float32)
    mag = rng.uniform(0.5, 1.5, n).astype(np.float32) if with_mag else None
    return w, packed, np.float32(ws), codes, x, q, s, grad, mag


def _run(dev, c, want_dbias=True):
    w, packed, ws, _, x, q, s, grad, mag = c
    t = lambda a: None if a is None else torch.from_numpy(a).to(dev)
    got = ops.bitlinear_ste_backward(x, q, s, t(w), t(packed.view(np.int32)), float(ws), t(grad),
                                     False, t(mag), want_dbias)
    return {key: v.cpu().numpy() for key, v in got.items()}


def _want(c):
    w, _, ws, codes, _, q, s, grad, mag = c
    q, s = q.cpu().numpy().astype(np.float64), s.cpu().numpy().astype(np.float64)
    g = grad.astype(np.float64)
    gp = g if mag is None else g * mag
    keep = np.abs(w / np.float32(ws + np.float32(1e-8))) <= 1.0
    with np.errstate(invalid="ignore"):
        pre = (q @ codes.T) * (s * float(ws))[:, None]
        out = {"dW": (gp.T @ (q * s[:, None])), "dx": gp @ (codes * float(ws)),
               "dmag": (g * pre).sum(0), "dbias": g.sum(0)}
    out["dW"] = np.where(keep, out["dW"], 0.0)
    return out


@pytest.mark.parametrize("m,k,n", [(1, 16, 4), (31, 16, 36), (32, 256, 128), (33, 272, 132),
                                   (64, 240, 124), (96, 528, 260), (129, 512, 64), (200, 1040, 384)])
@pytest.mark.parametrize("with_mag", [True, False])
def test_ste_sums_within_float_sum_bound(dev, m, k, n, with_mag):
    """Gradients over twelve binades either way, so that the small pieces count."""
    c = _case(dev, m, k, n, with_mag, 7 * m + k + n, spread=4096.0)
    got, want = _run(dev, c), _want(c)
    _, _, ws, codes, _, q, s, grad, mag = c
    absw = list(c)
    absw[7], absw[3] = np.abs(grad), np.abs(codes)
    absw[5] = q.abs()
    absw[0] = np.zeros_like(c[0])  # no clip
    size = _want(tuple(absw))
    terms = {"dW": m + 4, "dx": n + 4, "dmag": m + k + 8, "dbias": m}
    if with_mag:
        # dmag adds T * (sum over rows of grad * as * q): its terms' magnitudes are those of
        # sum_k |T| sum_i |grad| as |q|
        a = np.abs(q.cpu().numpy().astype(np.float64)) * s.cpu().numpy().astype(np.float64)[:, None]
        size["dmag"] = float(ws) * ((np.abs(grad).astype(np.float64).T @ a) * np.abs(codes)).sum(1)
    for key, g in got.items():
        err = np.abs(g.astype(np.float64) - want[key])
        assert np.all(err <= terms[key] * U * size[key] + 1e-37), key


@pytest.mark.parametrize("m,n", [(70, 40), (64, 132)])
def test_ste_infinities_and_nan_stay_where_they_are(dev, m, n):
    k = 272
    c = _case(dev, m, k, n, True, m + n)
    grad = c[7]
    grad[3, 5], grad[40, 6], grad[m - 1, n - 1], grad[12, 9] = np.inf, -np.inf, np.inf, np.nan
    got, want = _run(dev, c), _want(c)
    for key, g in got.items():
        np.testing.assert_array_equal(np.isnan(g), np.isnan(want[key]), err_msg=key)
        inf = np.isinf(want[key])
        np.testing.assert_array_equal(g[inf], want[key][inf].astype(np.float32), err_msg=key)
        assert np.array_equal(np.isinf(g), inf), key


@pytest.mark.parametrize("m,k,n,out,over", [
    (300, 384, 384, "dx", "grad"), (384, 272, 384, "dW", "grad"), (256, 528, 260, "dW", "grad"),
    (300, 272, 260, "dbias", "grad"), (300, 272, 260, "dmag", "grad"),
    (300, 272, 260, "dbias", "mag"), (300, 272, 260, "dmag", "mag"), (300, 528, 260, "dx", "mag"),
    (300, 528, 260, "dW", "mag"), (384, 272, 384, "dx", "w"), (300, 272, 260, "dx", "q"),
    (300, 272, 260, "dx", "s"), (300, 272, 260, "dW", "w")])
@pytest.mark.parametrize("odd", [False, True])
def test_ste_outputs_over_inputs(dev, m, k, n, out, over, odd):
    """An output laid over an input gives the bits of one apart, also where gradients are not finite
    (dmag reads them again then)."""
    w, packed, ws, _, x, q, s, grad, mag = _case(dev, m, k, n, True, m + k + n)
    if odd:
        grad[3, 5], grad[40, 6], grad[m - 1, n - 1] = np.inf, -np.inf, np.nan
    t = lambda a: torch.from_numpy(a).to(dev)
    nbytes = int(lib().nsosx_bitlinear_ste_backward_workspace(m, k, n, 0))

    def run(lay):
        shapes = {"dx": (m, k), "dW": (n, k), "dmag": (n,), "dbias": (n,)}
        src = {"q": q.contiguous(), "s": s.contiguous(), "w": t(w), "grad": t(grad), "mag": t(mag)}
        bufs = {key: torch.empty(shape, device=dev) for key, shape in shapes.items()}
        if lay:  # one block of memory that holds both from its first byte
            a, b = src[over], bufs[out]
            block = torch.empty(max(a.numel() * a.element_size(), b.numel() * 4), dtype=torch.uint8, device=dev)
            src[over] = block[:a.numel() * a.element_size()].view(a.dtype).view(a.shape).copy_(a)
            bufs[out] = block[:b.numel() * 4].view(torch.float32).view(b.shape)
        p = lambda v: v.data_ptr()
        work = torch.empty(nbytes, dtype=torch.uint8, device=dev)
        call("nsosx_bitlinear_ste_backward", None, 0, p(src["q"]), p(src["s"]), p(src["w"]),
             p(packed_t), float(ws), m, k, n, 0, p(src["mag"]), p(src["grad"]), p(bufs["dx"]), p(bufs["dW"]),
             p(bufs["dmag"]), p(bufs["dbias"]), p(work), None)
        torch.cuda.synchronize()
        return bufs

    packed_t = t(packed.view(np.int32))
    want, got = run(False), run(True)
    for key in want:
        np.testing.assert_array_equal(got[key].cpu().numpy(), want[key].cpu().numpy(), err_msg=key)


def test_ste_dmag_with_row_scales_not_finite(dev):
    """A row whose act_scale is infinite or NaN leaves in dmag what the definition gives."""
    m, k, n = 70, 272, 40
    c = list(_case(dev, m, k, n, True, 5))
    c[6] = c[6].clone()
    c[6][3], c[6][69] = np.inf, np.inf
    got, want = _run(dev, c)["dmag"], _want(c)["dmag"]
    np.testing.assert_array_equal(got, want.astype(np.float32))
    assert np.isinf(got).any()
    c[6][5] = np.nan
    assert np.isnan(_run(dev, c)["dmag"]).all()


@pytest.mark.parametrize("kind", ["+inf", "inf", "nan"])
def test_ste_time_when_every_gradient_overflowed(dev, kind):
    """A step whose gradients overflowed (as under loss scaling) takes about its usual time: the
    tiles' second pass over the infinities and a short walk per column, not M * K steps of one
    thread (290 times the usual time at a quarter of this size)."""
    m, k, n = 1024, 512, 512
    w, packed, ws, _, x, q, s, grad, mag = _case(dev, m, k, n, True, 11)
    t = lambda a: torch.from_numpy(a).to(dev)
    wd, pd, md = t(w), t(packed.view(np.int32)), t(mag)
    usual = t(grad)
    bad = {"+inf": torch.full_like(usual, np.inf), "nan": torch.full_like(usual, np.nan),
           "inf": torch.where(usual > 0, np.inf, -np.inf).to(torch.float32)}[kind]

    def us(g):
        run = lambda: ops.bitlinear_ste_backward(x, q, s, wd, pd, float(ws), g, False, md, True)
        run()
        best = np.inf
        for _ in range(5):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            run()
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        return best

    assert us(bad) < 10 * us(usual)


@pytest.mark.parametrize("e", [-126, -118, -110, -100, 0, 60, 84])
@pytest.mark.parametrize("with_mag", [True, False])
def test_ste_precision_at_every_magnitude(dev, with_mag, e):
    """Gradients of 2^e: their pieces hold every bit, of small ones too (a denormal bf16 reads as
    zero in the matrix cores), and sums that overflow only on the way come out as they are.  The
    bound is the float sum's, as above; results below 2^-126 round to multiples of 2^-149."""
    m, k, n = 200, 272, 132
    c = list(_case(dev, m, k, n, with_mag, 17, spread=16.0))
    with np.errstate(under="ignore"):
        c[7] = np.ldexp(c[7], e).astype(np.float32)
    c[6] = torch.full_like(c[6], 2.0 ** 12)  # (keeps dW and dmag normal for the smallest)
    got, want = _run(dev, tuple(c)), _want(tuple(c))
    absw = list(c)
    absw[7], absw[3], absw[5], absw[0] = np.abs(c[7]), np.abs(c[3]), c[5].abs(), np.zeros_like(c[0])
    size = _want(tuple(absw))
    terms = {"dW": m + 4, "dx": n + 4, "dmag": m + k + 8, "dbias": m}
    if with_mag:
        a = np.abs(c[5].cpu().numpy().astype(np.float64)) * c[6].cpu().numpy().astype(np.float64)[:, None]
        size["dmag"] = float(c[2]) * ((np.abs(c[7]).astype(np.float64).T @ a) * np.abs(c[3])).sum(1)
    for key, g in got.items():
        err = np.abs(g.astype(np.float64) - want[key])
        # (a product that underflows is rounded to 2^-149 before it is added)
        assert np.all(err <= terms[key] * (U * size[key] + 2.0 ** -149)), key
