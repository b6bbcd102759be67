"""RMS_PERI + int8 codes of few rows (a workgroup per row, the in-order sum taken from composed
runs): codes and scales bit for bit against the oracle's sequential sum, on rows built to hit the
runs' edges -- ties at every addition, sums that sit on a binade's end, jumps over several
binades, zeros, denormals, and values that are not finite."""
import numpy as np
import pytest
import torch

from reimagined_amd import ops
from reimagined_amd._lib import call

pytestmark = pytest.mark.gpu


def _rows(rng, k, bf16):
    n = lambda *s: rng.standard_normal(s if s else k)
    rows = [n(), n() * 1e-3, np.ones(k), np.full(k, 2.0 ** -12), np.full(k, 3.0 * 2.0 ** -13)]
    # heavy tails: the sum jumps binades at random places
    rows += [np.exp(4.0 * n()) * np.sign(n()), rng.standard_cauchy(k)]
    # squares that are exact halves of an ulp of the sum from the second element on
    tie = np.full(k, 2.0 ** -12); tie[0] = 1.0
    rows.append(tie)
    tie = np.full(k, 2.0 ** -12 * 1.5); tie[0] = 1.0
    rows.append(tie)
    # the sum stands just below a power of two, then crosses by one ulp at the row's end
    edge = np.zeros(k); edge[0] = np.sqrt(1.0 - 2.0 ** -20); edge[1:] = 2.0 ** -13
    rows.append(edge)
    up = np.zeros(k); up[k // 2:] = 1.0
    rows.append(up)
    rows.append(np.zeros(k))
    jump = np.full(k, 2.0 ** -10); jump[k // 3] = 300.0; jump[-1] = 1e4
    rows.append(jump)
    rows.append(np.full(k, 1e-22))                       # denormal squares and sums
    rows.append(np.where(np.arange(k) % 7 == 0, 1e-3, 1e-22))
    rows.append(np.exp2(np.linspace(-40, 40, k)))        # a crossing every few elements
    rows.append(np.exp2(np.linspace(40, -40, k)))
    rows.append(n() * 1e18)                              # sums near the top of the range
    rows += [n() * (0.5 + 0.1 * i) for i in range(15)]
    x = np.stack(rows).astype(np.float32)
    return torch.from_numpy(x).to(torch.bfloat16).float().numpy() if bf16 else x


@pytest.mark.parametrize("k", [8, 16, 64, 504, 512, 520, 768, 1024, 1032, 2048, 2560, 4088, 4096])
@pytest.mark.parametrize("bf16", [True, False])
def test_few_rows_rms_codes_bit_exact(dev, orc, k, bf16):
    x = _rows(np.random.default_rng(k), k, bf16)
    xd = torch.from_numpy(x).to(torch.bfloat16 if bf16 else torch.float32).to(dev)
    q, s = ops.quantize_activations_bitnet(xd, 8, rms_input=True)
    wq, ws = orc.quantize_act(orc.rmsnorm(x), 8)
    np.testing.assert_array_equal(s.cpu().numpy(), ws)
    np.testing.assert_array_equal(q.cpu().numpy(), wq)


@pytest.mark.parametrize("k", [512, 1024, 4096])
def test_few_rows_equal_many_rows(dev, k):
    """The same rows through this launch and through the passes that take many rows, also with
    infinities and NaN (whose codes and scales both define as the arithmetic falls)."""
    rng = np.random.default_rng(k + 1)
    x = rng.standard_normal((64, k)).astype(np.float32)
    x[3, 5], x[4, k - 1], x[5, 0], x[6, 7] = np.inf, -np.inf, np.nan, 3e38
    x[7] = np.inf
    x[8, :9] = [np.inf, np.nan, 0, 0, 1, 1, 1, 1, np.inf]
    few = torch.from_numpy(x).to(dev)
    q, s = ops.quantize_activations_bitnet(few, 8, rms_input=True)
    many = torch.cat([few, torch.ones((40000, k), device=dev)])
    wq, ws = ops.quantize_activations_bitnet(many, 8, rms_input=True)
    np.testing.assert_array_equal(q.cpu().numpy(), wq[:64].cpu().numpy())
    np.testing.assert_array_equal(s.cpu().numpy(), ws[:64].cpu().numpy())


@pytest.mark.parametrize("bf16,k,rows", [(True, 2048, 3072), (True, 2560, 2560), (True, 2600, 3072), (False, 896, 4096),
                                         (False, 1024, 6144), (False, 1280, 3584), (False, 1288, 6144)])
def test_last_rows_of_the_one_launch_and_first_of_the_passes(dev, bf16, k, rows):
    """Both sides of the row limit leave the bits of the rows by themselves."""
    x = torch.randn((rows + 1, k), device=dev).to(torch.bfloat16 if bf16 else torch.float32)
    x[-1, : k // 2] = 0
    want_q, want_s = ops.quantize_activations_bitnet(x[-65:].contiguous(), 8, rms_input=True)
    for part in (x[1:].contiguous(), x):
        q, s = ops.quantize_activations_bitnet(part, 8, rms_input=True)
        assert torch.equal(q[-65:], want_q) and torch.equal(s[-65:], want_s)


@pytest.mark.parametrize("k,n", [(64, 48), (512, 33), (1024, 4096), (2048, 1000), (2112, 64),
                                 (4096, 256)])
@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("rms", [True, False])
def test_one_row_forward_equals_quantize_then_gemv(dev, orc, k, n, bf16, rms):
    """The one-launch forward of a row, bit for bit the oracle's quantization and affine."""
    rng = np.random.default_rng(k + n)
    packed, ws, codes = orc.pack_weights(rng.standard_normal((n, k)).astype(np.float32))
    mag = rng.uniform(0.5, 1.5, n).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    pk = torch.from_numpy(packed.view(np.int32)).to(dev)
    t = lambda a: torch.from_numpy(a).to(dev)
    for row in _rows(rng, k, bf16)[[0, 5, 7, 11, 12, 15]]:
        x = torch.from_numpy(row[None]).to(torch.bfloat16 if bf16 else torch.float32).to(dev)
        y = ops.bitnet_gemm_158bit_gpu(x, pk, ws, 1, k, n, magnitude=t(mag), bias=t(bias),
                                       rms_input=rms)
        want = orc.bitlinear_forward(row[None], packed, ws, n, rms_input=rms, magnitude=mag,
                                     bias=bias)
        np.testing.assert_array_equal(y.cpu().numpy(), want)


@pytest.mark.parametrize("k,n", [(512, 512), (1024, 1000), (4096, 4096)])
@pytest.mark.parametrize("rms", [True, False])
def test_one_row_forward_keeps_the_codes_and_runs_in_place(dev, orc, k, n, rms):
    """The workspaces hold the row's codes and scale afterwards, as a backward reads them, and y
    may lie over x."""
    rng = np.random.default_rng(k)
    packed, ws, _ = orc.pack_weights(rng.standard_normal((n, k)).astype(np.float32))
    pk = torch.from_numpy(packed.view(np.int32)).to(dev)
    x = torch.randn((1, k), device=dev)
    want_q, want_s = ops.quantize_activations_bitnet(x, 8, rms_input=rms)
    want = ops.ternary_gemm(want_q, want_s, pk, ws, n)
    q = torch.zeros((1, k), dtype=torch.int8, device=dev)
    s, r = torch.zeros(1, device=dev), torch.zeros(1, device=dev)
    buf = torch.zeros(max(k, n), device=dev)
    for y in (torch.empty(n, device=dev), buf):
        buf[:k] = x[0]
        call("nsosx_bitlinear_forward", buf.data_ptr(), 0, pk.data_ptr(), ws, 1, k, n, 8, int(rms), None,
             None, y.data_ptr(), 0, q.data_ptr(), s.data_ptr(), r.data_ptr(), None)
        torch.cuda.synchronize()
        assert torch.equal(q, want_q) and torch.equal(s, want_s)
        assert torch.equal(y[:n], want.view(-1))


def _one_row_forward(dev, k, n, rms, pk, ws, x, over=None):
    """The C entry on buffers of its own, or with over = (a, b): b lies over a from its first byte."""
    size = {"x": 4 * k, "y": 4 * n, "q": k, "s": 4, "r": 4}
    mem = {key: torch.zeros(max(size.values()), dtype=torch.uint8, device=dev) for key in size}
    if over:
        mem[over[1]] = mem[over[0]]
    mem["x"][:4 * k] = x.view(torch.uint8).view(-1)
    p = {key: v.data_ptr() for key, v in mem.items()}
    call("nsosx_bitlinear_forward", p["x"], 0, pk.data_ptr(), ws, 1, k, n, 8, int(rms), None, None,
         p["y"], 0, p["q"], p["s"], p["r"], None)
    torch.cuda.synchronize()
    return {key: v[:size[key]] for key, v in mem.items()}


@pytest.mark.parametrize("k,n", [(512, 512), (1024, 1000), (4096, 4096)])
@pytest.mark.parametrize("rms", [True, False])
def test_one_row_forward_keeps_codes_scale_and_rms(dev, orc, k, n, rms):
    """The workspaces hold the row's codes, scale and 1 / rms afterwards, as a backward reads them;
    buffers that lie over one another leave what one apart from the other leaves."""
    rng = np.random.default_rng(k)
    packed, ws, _ = orc.pack_weights(rng.standard_normal((n, k)).astype(np.float32))
    pk = torch.from_numpy(packed.view(np.int32)).to(dev)
    x = torch.randn((1, k), device=dev)
    want = {"q": torch.zeros((1, k), dtype=torch.int8, device=dev), "s": torch.zeros(1, device=dev),
            "r": torch.zeros(1, device=dev)}
    call("nsosx_quantize_act_i8", x.data_ptr(), 0, 1, k, 8, int(rms), want["q"].data_ptr(),
         want["s"].data_ptr(), want["r"].data_ptr(), None)
    want["y"] = ops.ternary_gemm(want["q"], want["s"], pk, ws, n)
    want = {key: v.contiguous().view(torch.uint8).view(-1) for key, v in want.items()}
    got = _one_row_forward(dev, k, n, rms, pk, ws, x)
    for key in want:
        assert torch.equal(got[key], want[key]), key
    # the later of two stores stands: r, then s, then q, then y
    for a, b in (("x", "y"), ("x", "q"), ("x", "s"), ("x", "r"), ("r", "s"), ("r", "y"), ("r", "q")):
        got = _one_row_forward(dev, k, n, rms, pk, ws, x, (a, b))
        for key in ("y", "q", "s", "r"):
            if not (key == "r" and (a == "r" or not rms)):
                assert torch.equal(got[key], want[key]), (a, b, key)


@pytest.mark.parametrize("k", [512, 1024, 2048, 4096])
def test_rows_of_zeros_and_overflow_take_the_usual_time(dev, k):
    """Padding rows, rows that start with zeros and denormal squares cost no more than ordinary rows
    (added thread by thread 4 to 13 times as much).  A row with an infinity or a sum that doubles
    every few elements is one chain of K additions, 9 cycles each: at K = 4096 20 us, 2.6 times
    the ordinary call."""
    m = 64
    rows = {"usual": torch.randn((m, k), device=dev)}
    rows["zero"] = torch.zeros((m, k), device=dev)
    rows["late"] = rows["zero"].clone()
    rows["late"][:, k - 8:] = 1.0
    rows["tiny"] = rows["usual"] * 1e-22
    rows["inf"] = rows["usual"].clone()
    rows["inf"][:, 0] = np.inf
    rows["ramp"] = torch.exp2(torch.linspace(-40, 40, k, device=dev)).expand(m, k).contiguous()

    def us(x):
        q, s, r = (torch.empty((m, k), dtype=torch.int8, device=dev), torch.empty(m, device=dev),
                   torch.empty(m, device=dev))
        run = lambda: call("nsosx_quantize_act_i8", x.data_ptr(), 0, m, k, 8, 1, q.data_ptr(),
                           s.data_ptr(), r.data_ptr(), torch.cuda.current_stream().cuda_stream)
        run()
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            for _ in range(20):
                run()
        best = np.inf
        for _ in range(5):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            g.replay()
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        return best

    usual = us(rows["usual"])
    for name, most in (("zero", 2), ("late", 2), ("tiny", 2), ("inf", 4), ("ramp", 4)):
        assert us(rows[name]) < most * usual, name
