"""The scan at one A per head and d_state 32 .. 64 with the chunk length the library picks, against
the float64 recurrence on both sides of chunk edges, and against the unchunked scan where the
inputs are not finite.  Tolerance: the scan's own 1e-4 relative / 1e-5 absolute."""
import numpy as np
import pytest
import torch

from reimagined_amd import ops
from reimagined_amd._lib import call

pytestmark = pytest.mark.gpu


def _inputs(dev, lengths, H, N, G, seed, dtype, dt_mean=-2.0):
    rng = np.random.default_rng(seed)
    T = int(sum(lengths))
    t = lambda a, d=torch.float32: torch.from_numpy(np.ascontiguousarray(a, np.float32)).to(d).to(dev)
    return {"x": t(rng.standard_normal((T, H * 64)), dtype), "dt": t(rng.normal(dt_mean, 1.0, (T, H)), dtype),
            "a_log": t(rng.standard_normal(H)), "B": t(rng.normal(0, 0.5, (T, G * N)), dtype),
            "C": t(rng.normal(0, 0.5, (T, G * N)), dtype), "D": t(rng.standard_normal(H)),
            "conv_w": t(rng.standard_normal((H * 64, 4)) * 0.5), "conv_b": t(rng.standard_normal(H * 64) * 0.1),
            "init": t(rng.normal(0, 0.3, (len(lengths), H * 64, N))),
            "cu": torch.from_numpy(np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)).to(dev)}


def _run(d, H, N, G, width, init, chunk):
    args = (d["dt"], d["a_log"], d["B"], d["C"], d["D"], None, d["cu"], H, 64, N, G)
    kw = dict(initial_state=d["init"] if init else None, chunk_tokens=chunk)
    if width == 0:
        return ops.selective_scan_fwd(d["x"], *args, **kw)
    return ops.conv_scan_fwd(d["x"], d["conv_w"][:, :width].contiguous(), d["conv_b"], *args, **kw)


def _float64(d, lengths, H, N, G, width, init):
    x, cu = d["x"].double(), d["cu"].tolist()
    out, fin = torch.zeros_like(x), torch.zeros(len(lengths), H * 64, N, dtype=torch.float64, device=x.device)
    a = -torch.exp(d["a_log"].double()).repeat_interleave(64)[:, None]
    delta = torch.nn.functional.softplus(d["dt"].double(), threshold=1e9).repeat_interleave(64, 1)
    group = torch.arange(H, device=x.device) * G // H
    for s in range(len(lengths)):
        xs = x[cu[s]:cu[s + 1]]
        if width:
            pad = torch.cat([xs.new_zeros(width - 1, xs.shape[1]), xs])
            acc = sum(pad[j:j + len(xs)] * d["conv_w"][:, j].double() for j in range(width))
            xs = torch.nn.functional.silu(acc + d["conv_b"].double())
        h = d["init"][s].double().clone() if init else fin[s].clone()
        for i in range(len(xs)):
            t = cu[s] + i
            b, c = (d[k][t].double().view(G, N)[group].repeat_interleave(64, 0) for k in ("B", "C"))
            h = h * torch.exp(delta[t][:, None] * a) + (delta[t] * xs[i])[:, None] * b
            out[t] = (h * c).sum(1) + d["D"].double().repeat_interleave(64) * xs[i]
        fin[s] = h
    return out, fin


@pytest.mark.parametrize("lengths", [[129], [160, 127, 128, 129], [400, 0, 1], [97, 256], [31, 513, 32, 33]])
@pytest.mark.parametrize("H,N,G,width,init", [(2, 64, 1, 4, False), (4, 48, 2, 4, True), (2, 32, 2, 0, True),
                                              (1, 64, 1, 2, True), (3, 32, 1, 1, False)])
def test_wide_scan_matches_float64(dev, lengths, H, N, G, width, init):
    d = _inputs(dev, lengths, H, N, G, sum(lengths) + N, torch.float32)
    y, fin = _run(d, H, N, G, width, init, -1)
    wy, wf = _float64(d, lengths, H, N, G, width, init)
    torch.testing.assert_close(y.double(), wy, rtol=1e-4, atol=1e-5)
    torch.testing.assert_close(fin.double(), wf, rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("dt_mean", [-8.0, -2.0, 3.0])
def test_wide_scan_no_less_exact_than_sequential(dev, dt_mean):
    """Slow, ordinary and strong decays (a chunk's summed exponents reach -1e5)."""
    lengths, H, N, G = [700, 257, 64], 8, 64, 1
    d = _inputs(dev, lengths, H, N, G, 11, torch.float32, dt_mean)
    wy, wf = _float64(d, lengths, H, N, G, 4, True)
    err = lambda a, b: ((a.double() - b).norm() / b.norm()).item()
    got, seq = (_run(d, H, N, G, 4, True, c) for c in (-1, 0))
    for a, b, w in ((got[0], seq[0], wy), (got[1], seq[1], wf)):
        assert err(a, w) <= max(1.2 * err(b, w), 2e-7), (dt_mean, err(a, w), err(b, w))


def test_wide_scan_bf16(dev):
    lengths, H, N, G = [230, 75], 4, 64, 1
    d = _inputs(dev, lengths, H, N, G, 5, torch.bfloat16)
    y, fin = _run(d, H, N, G, 4, True, -1)
    wy, wf = _float64(d, lengths, H, N, G, 4, True)
    torch.testing.assert_close(y.double(), wy, rtol=2.0 ** -8, atol=1e-4)  # one bf16 rounding
    torch.testing.assert_close(fin.double(), wf, rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("what", ["x", "B", "C", "dt", "init", "huge"])
def test_wide_scan_keeps_what_is_not_finite(dev, what):
    lengths, H, N, G = [200, 140], 2, 64, 1
    d = _inputs(dev, lengths, H, N, G, 8, torch.float32)
    if what == "init":
        d["init"][1, 70, 3] = float("inf")
    elif what == "huge":
        d["x"][40, 5], d["B"][40, 2] = 3e38, 30.0
    else:
        d[what][150, 1] = float("nan")
        d[what][20, 0] = float("inf") if what != "dt" else 50.0
    got, seq = (_run(d, H, N, G, 4, True, c) for c in (-1, 0))
    for a, b in zip(got, seq):
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.isinf(a), torch.isinf(b))
        ok = torch.isfinite(b)
        # (huge: sums of 1e38 terms that cancel, exact to the terms' size and not the sum's)
        atol = 1e-5 if what != "huge" else 1e-6 * b[ok].abs().max().item()
        torch.testing.assert_close(a[ok], b[ok], rtol=1e-4, atol=atol)


def test_wide_scan_refuses_a_short_stride_and_runs_in_place(dev):
    """A row stride below H * P stays refused, and y over x gives what a buffer of its own does."""
    lengths, H, N = [300, 129], 2, 64
    d = _inputs(dev, lengths, H, N, 1, 4, torch.float32)
    T, D = sum(lengths), H * 64
    ws = torch.empty(int(ops.lib().nsosx_scan_fwd_workspace(2, T, H, 64, N, -1)), dtype=torch.uint8, device=dev)
    p = lambda k: d[k].data_ptr()

    def run(stride, y):
        call("nsosx_scan_fwd_planned", p("x"), stride, None, None, 0, p("dt"), p("a_log"), 0, p("B"), p("C"),
             p("D"), None, 0, p("cu"), 2, T, H, 64, N, 1, 0, None, None, y.data_ptr(), -1, ws.data_ptr(), None)
        torch.cuda.synchronize()

    y = torch.empty((T, D), device=dev)
    with pytest.raises(Exception, match="stride"):
        run(D - 64, y)
    run(D, y)
    run(D, d["x"])
    torch.testing.assert_close(d["x"], y, rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("N,G,width,init,dtype", [(64, 1, 4, False, torch.float32), (64, 2, 0, True, torch.bfloat16),
                                                  (48, 1, 2, True, torch.float32), (32, 1, 4, True, torch.float32)])
@pytest.mark.parametrize("lengths", [[1025, 300], [2177], [129, 512]])
def test_wide_scan_bits_are_the_recurrences(dev, lengths, N, G, width, init, dtype):
    """The chunk length the library picks (here its least, 64 tokens) changes the carried states and
    nothing else: the same bits as that length asked for.  A last-bit change of y moves int8 codes
    of the projection behind the scan, which is 2e-4 of a block's output."""
    H = 4
    d = _inputs(dev, lengths, H, N, G, sum(lengths) + 3 * N, dtype)
    for a, b in zip(_run(d, H, N, G, width, init, -1), _run(d, H, N, G, width, init, 64)):
        assert torch.equal(a, b)
