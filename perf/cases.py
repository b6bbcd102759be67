"""The work a user of this package has it do, as cases that can be timed and compared.

Every case goes through the package's public entry points (reimagined_amd.layers and
reimagined_amd.ops) as a serving or training program calls them, over seven kinds:

  linear       BitLinear.forward: RMS norm, int8 quantization, ternary GEMV / GEMM
  layer        HybridMambaLayer.forward over a packed ragged batch, with final states
  block        HybridBlock.forward: norms, Mamba layer, routed experts, residuals
  moe          MoEFFN.forward, or .decode for a few rows
  mamba2       Mamba2Block.forward over a packed ragged batch, with final states
  mamba2_step  Mamba2Block.step: one decode token per row, states updated in place
  scan_step    ops.selective_scan_step: the recurrence of one decode token per row
  train        a BitLinear training step: forward, then the straight-through backward

Sizes are those of the configurations in reimagined_amd/workloads.py and bench.py (d_model
768 / 1024 / 2048, expansion 2, 4x feed-forward, 8 experts top-2, d_state 16 or the
faithful block's default 64, sequences of 64 to 2048 tokens); draw() spreads row counts,
sequence counts and widths over the ranges between them.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from reimagined_amd import layers, ops

_DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def listed():
    return [
        # one token of one user through a projection: launch latency and one weight read
        dict(name="linear_decode", kind="linear", rows=1, k=1024, n=4096, dtype="bf16",
             affine=False),
        # a decode batch of 64 users through a feed-forward sized projection
        dict(name="linear_batch", kind="linear", rows=64, k=2048, n=8192, dtype="bf16",
             affine=False),
        # a short prompt through the smallest configuration's 768 x 768 projection, in
        # float32 with the magnitude and bias that trained checkpoints carry
        dict(name="linear_prompt_f32", kind="linear", rows=300, k=768, n=768, dtype="f32",
             affine=True),
        # prefill of 4096 tokens through the wide projection
        dict(name="linear_prefill", kind="linear", rows=4096, k=2048, n=8192, dtype="bf16",
             affine=False),
        # the headline: prefill of a packed batch of 32 ragged prompts through a Mamba layer
        dict(name="layer_ragged", kind="layer", seqs=32, lo=64, hi=2048, d_model=1024,
             d_state=16, dtype="bf16"),
        # one user's prompt through a whole hybrid block (Mamba core + experts)
        dict(name="block_prompt", kind="block", seqs=1, lo=1500, hi=1500, d_model=1024,
             d_state=16, experts=8, top_k=2, dtype="bf16"),
        # prefill of the routed feed-forward
        dict(name="moe_prefill", kind="moe", rows=8192, d_model=1024, d_ff=4096, experts=8,
             top_k=2, sparse=False, dtype="bf16"),
        # a decode batch of 48 users through the routed feed-forward
        dict(name="moe_batch", kind="moe", rows=48, d_model=1024, d_ff=4096, experts=8,
             top_k=2, sparse=False, dtype="bf16"),
        # prefill of the faithful Mamba-2 block at the model's default state size, float32
        dict(name="mamba2_prefill", kind="mamba2", seqs=8, lo=64, hi=2048, d_model=1024,
             heads=32, d_state=64, dtype="f32"),
        # one decode token of 16 users through the same block
        dict(name="mamba2_step", kind="mamba2_step", rows=16, d_model=1024, heads=32,
             d_state=64, dtype="f32"),
        # one decode token of 256 sequences through the Mamba-1 recurrence
        dict(name="scan_step", kind="scan_step", rows=256, channels=2048, d_state=16,
             dtype="bf16"),
        # a training step of an in_proj sized projection over 4096 tokens
        dict(name="train_step", kind="train", rows=4096, k=1024, n=4096, rms=True, affine=True,
             dtype="f32"),
    ]


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm, odd ones among them."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "layer", "layer", "block", "moe", "moe",
                       "mamba2", "mamba2_step", "scan_step", "train"])
    dtype = rng.choice(["bf16", "bf16", "f32"])
    if kind == "linear":
        k = rng.choice([512, 768, 1024, 1536, 2048, 2560, 4096])
        n = 16 * _spread(rng, 32, 512)
        most = 4096 * 2048 * 8192 // (k * n)
        return dict(kind=kind, rows=_spread(rng, 1, min(8192, most)), k=k, n=n, dtype=dtype,
                    affine=rng.random() < 0.4)
    if kind in ("layer", "block"):
        d_model = rng.choice([512, 768, 1024])
        seqs = _spread(rng, 1, 16 if kind == "layer" else 4)
        lo = _spread(rng, 16, 512)
        c = dict(kind=kind, seqs=seqs, lo=lo, hi=lo + _spread(rng, 16, 1024), d_model=d_model,
                 d_state=16, dtype=dtype)
        if kind == "block":
            c.update(experts=rng.choice([4, 8]), top_k=rng.choice([1, 2]))
        return c
    if kind == "moe":
        rows = _spread(rng, 1, 6000)
        return dict(kind=kind, rows=rows, d_model=rng.choice([512, 768, 1024]), d_ff=4096,
                    experts=rng.choice([4, 8, 16]), top_k=rng.choice([1, 2, 2]),
                    sparse=rows <= 8, dtype=dtype)
    if kind == "mamba2":
        lo = _spread(rng, 16, 512)
        heads = rng.choice([16, 24, 32])
        return dict(kind=kind, seqs=_spread(rng, 1, 8), lo=lo, hi=lo + _spread(rng, 16, 1024),
                    d_model=32 * heads, heads=heads, d_state=rng.choice([16, 32, 64, 64]),
                    dtype=rng.choice(["f32", "f32", "bf16"]))
    if kind == "mamba2_step":
        heads = rng.choice([16, 24, 32])
        return dict(kind=kind, rows=_spread(rng, 1, 64), d_model=32 * heads, heads=heads,
                    d_state=rng.choice([16, 64]), dtype="f32")
    if kind == "scan_step":
        return dict(kind=kind, rows=_spread(rng, 1, 256), channels=rng.choice([1024, 1536, 2048]),
                    d_state=16, dtype=dtype)
    k = rng.choice([512, 768, 1024])
    n = 16 * _spread(rng, 32, 256)
    return dict(kind="train", rows=_spread(rng, 64, 4096), k=k, n=n, rms=rng.random() < 0.7,
                affine=rng.random() < 0.6, dtype="f32")


# ---- inputs ---------------------------------------------------------------------

def _offsets(case):
    """cu_seqlens of a ragged batch: lengths uniform in [lo, hi], fixed by the case so that its
    outputs have one shape whatever the seed of the values."""
    rng = np.random.default_rng([case["seqs"], case["lo"], case["hi"]])
    lengths = rng.integers(case["lo"], case["hi"] + 1, size=case["seqs"])
    return np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)


def _data(case, seed):
    """The case's inputs and float weights, from the seed alone, as a dict of tensors on the
    GPU (activations in the case's dtype).  Latent weights are N(0, 0.02), activations N(0, 1),
    raw deltas around softplus^-1 of 0.1, B and C N(0, 1/16), A_log N(0, 1)."""
    g = torch.Generator("cuda").manual_seed(seed)
    dt = _DTYPES[case["dtype"]]

    def normal(*shape, std=1.0, mean=0.0, dtype=torch.float32):
        return (torch.randn(shape, generator=g, device="cuda") * std + mean).to(dtype)

    kind = case["kind"]
    d = {}
    if kind in ("linear", "train"):
        n, k = case["n"], case["k"]
        d["w"] = normal(n, k, std=0.02)
        d["x"] = normal(case["rows"], k, dtype=dt)
        d["mag"] = normal(n, std=0.1, mean=1.0) if case["affine"] else None
        d["bias"] = normal(n, std=0.1) if case["affine"] else None
        if kind == "train":
            d["grad"] = normal(case["rows"], n, std=1e-3)
        return d
    if kind in ("layer", "block", "mamba2"):
        d["cu"] = _offsets(case)
        rows = int(d["cu"][-1])
    else:
        rows = case["rows"]
    if kind in ("layer", "block"):
        dm, di, n = case["d_model"], 2 * case["d_model"], case["d_state"]
        d.update(w_in=normal(2 * di, dm, std=0.02), w_out=normal(dm, di, std=0.02),
                 conv_w=normal(di, 4, std=0.5), conv_b=normal(di, std=0.1),
                 a_log=normal(di, n), d_skip=normal(di), x=normal(rows, dm, dtype=dt),
                 dt=normal(rows, di, std=0.5, mean=-2.0, dtype=dt),
                 B=normal(rows, n, std=0.25, dtype=dt), C=normal(rows, n, std=0.25, dtype=dt))
    if kind == "block":
        dm, f = case["d_model"], 4 * case["d_model"]
        d.update(w_up=[normal(f, dm, std=0.02) for _ in range(case["experts"])],
                 w_down=[normal(dm, f, std=0.02) for _ in range(case["experts"])],
                 core_gamma=normal(dm, std=0.1, mean=1.0), ff_gamma=normal(dm, std=0.1, mean=1.0),
                 logits=normal(rows, case["experts"]))
    if kind == "moe":
        dm, f = case["d_model"], case["d_ff"]
        d.update(w_up=[normal(f, dm, std=0.02) for _ in range(case["experts"])],
                 w_down=[normal(dm, f, std=0.02) for _ in range(case["experts"])],
                 x=normal(rows, dm, dtype=dt), logits=normal(rows, case["experts"]))
    if kind in ("mamba2", "mamba2_step"):
        dm, h, n = case["d_model"], case["heads"], case["d_state"]
        inner, p = 64 * h, dm ** -0.5
        d.update(w_x=normal(inner, dm, std=0.02), w_z=normal(inner, dm, std=0.02),
                 w_B=normal(n, dm, std=p), w_C=normal(n, dm, std=p), w_dt=normal(h, dm, std=p),
                 w_out=normal(dm, inner, std=0.02), dt_bias=normal(h, std=0.5, mean=-2.0),
                 conv_w=normal(inner + 2 * n, 4, std=0.5), conv_b=normal(inner + 2 * n, std=0.1),
                 a_log=normal(h), d_skip=normal(h), norm_w=normal(inner, std=0.1, mean=1.0),
                 u=normal(rows, dm, dtype=dt))
        if kind == "mamba2_step":
            d.update(state=normal(rows, inner, n, std=0.1), ring=normal(rows, 3, inner + 2 * n))
    if kind == "scan_step":
        c, n = case["channels"], case["d_state"]
        d.update(x=normal(rows, c, dtype=dt), dt=normal(rows, c, std=0.5, mean=-2.0, dtype=dt),
                 a_log=normal(c, n), B=normal(rows, n, std=0.25, dtype=dt),
                 C=normal(rows, n, std=0.25, dtype=dt), D=normal(c), z=normal(rows, c, dtype=dt),
                 state=normal(rows, c, n, std=0.1))
    return d


def _host(t):
    return None if t is None else t.cpu().numpy()


def _layer_params(d):
    return {k: _host(d[k]) for k in ("w_in", "w_out", "conv_w", "conv_b", "a_log", "d_skip")}


def prepare(case, seed):
    kind, dt = case["kind"], _DTYPES[case["dtype"]]
    d = _data(case, seed)
    s = {"kind": kind, "case": case}
    if kind == "linear":
        s.update(x=d["x"], layer=layers.BitLinear(_host(d["w"]), magnitude=_host(d["mag"]),
                                                  bias=_host(d["bias"])))
        return s
    if kind == "train":
        packed, ws = ops.pack_ternary(_host(d["w"]))
        s.update(x=d["x"], w=d["w"], grad=d["grad"], mag=d["mag"], bias=d["bias"], ws=ws,
                 packed=torch.from_numpy(packed.view(np.int32)).cuda())
        return s
    if kind == "moe":
        s.update(x=d["x"], logits=d["logits"],
                 layer=layers.MoEFFN([_host(w) for w in d["w_up"]],
                                     [_host(w) for w in d["w_down"]], k=case["top_k"],
                                     hidden_dtype=dt))
        return s
    if kind == "scan_step":
        s.update({k: d[k] for k in ("x", "dt", "a_log", "B", "C", "D", "z", "state")})
        return s
    if kind in ("layer", "block"):
        cu = torch.from_numpy(d["cu"]).cuda()
        final = torch.zeros((case["seqs"], 2 * case["d_model"], case["d_state"]), device="cuda")
        s.update(x=d["x"], dt=d["dt"], B=d["B"], C=d["C"], cu=cu, final=final)
        if kind == "layer":
            s["layer"] = layers.HybridMambaLayer(_layer_params(d))
        else:
            s["logits"] = d["logits"]
            s["layer"] = layers.HybridBlock(
                _layer_params(d), [_host(w) for w in d["w_up"]], [_host(w) for w in d["w_down"]],
                k=case["top_k"], core_gamma=_host(d["core_gamma"]), ff_gamma=_host(d["ff_gamma"]))
        return s
    params = {k: _host(d[k]) for k in ("w_x", "w_z", "w_B", "w_C", "w_dt", "w_out", "dt_bias",
                                       "conv_w", "conv_b", "a_log", "d_skip", "norm_w")}
    params.update(H=case["heads"], P=64, N=case["d_state"], G=1)
    s.update(u=d["u"], layer=layers.Mamba2Block(params, dtype=dt))
    if kind == "mamba2":
        s["cu"] = torch.from_numpy(d["cu"]).cuda()
    else:
        s["dec"] = s["layer"].new_decode_state(case["rows"], "cuda")
        s["dec"]["state"].copy_(d["state"])
        s["dec"]["ring"].copy_(d["ring"])
    return s


def run(s):
    kind = s["kind"]
    if kind == "linear":
        return s["layer"].forward(s["x"])
    if kind == "layer":
        out = s["layer"].forward(s["x"], s["dt"], s["B"], s["C"], s["cu"], final_state=s["final"])
        return {"out": out, "final_state": s["final"]}
    if kind == "block":
        r = s["layer"].forward(s["x"], s["dt"], s["B"], s["C"], s["cu"], logits=s["logits"],
                               final_state=s["final"])
        return {"out": r["out"], "residual": r["residual"], "final_state": s["final"]}
    if kind == "moe":
        r = (s["layer"].decode if s["case"]["sparse"] else s["layer"].forward)(s["x"], s["logits"])
        return {k: r[k] for k in ("out", "weights", "selected")}
    if kind == "mamba2":
        r = s["layer"].forward(s["u"], s["cu"])
        return {"out": r["out"], "final_state": r["final_state"]}
    if kind == "mamba2_step":
        out = s["layer"].step(s["u"], s["dec"])
        return {"out": out, "state": s["dec"]["state"], "ring": s["dec"]["ring"]}
    if kind == "scan_step":
        c = s["case"]
        y = ops.selective_scan_step(s["x"], s["dt"], s["a_log"], s["B"], s["C"], s["D"], s["z"],
                                    s["state"], c["channels"], 1, c["d_state"], 1)
        return {"y": y, "state": s["state"]}
    rms = s["case"]["rms"]
    q, scale = ops.quantize_activations_bitnet(s["x"], 8, rms_input=rms)
    y = ops.ternary_gemm(q, scale, s["packed"], s["ws"], s["w"].shape[0], magnitude=s["mag"],
                         bias=s["bias"])
    grads = ops.bitlinear_ste_backward(s["x"], q, scale, s["w"], s["packed"], s["ws"], s["grad"],
                                       rms_input=rms, magnitude=s["mag"],
                                       want_dbias=s["bias"] is not None)
    return {"y": y, **grads}


# ---- what a pass cannot do without -----------------------------------------------

def work(case):
    kind = case["kind"]
    e = 2 if case["dtype"] == "bf16" else 4
    if kind == "linear":
        m, k, n = case["rows"], case["k"], case["n"]
        return {"bytes": m * k * e + n * k / 4 + m * n * e, "flops": 2.0 * m * k * n}
    if kind == "train":
        m, k, n = case["rows"], case["k"], case["n"]
        return {"bytes": 4.0 * (2 * m * k + 2 * n * k + 2 * m * n) + n * k / 4,
                "flops": 6.0 * m * k * n}
    if kind == "scan_step":
        r, c, n = case["rows"], case["channels"], case["d_state"]
        return {"bytes": 8.0 * r * c * n + 4 * r * c * e + 2 * r * n * e + 4 * c * n,
                "flops": 6.0 * r * c * n}

    def mamba(t, s, dm, n):
        di = 2 * dm
        return (t * (2 * dm + di + 2 * n) * e + 3 * dm * di / 4 + 4.0 * s * di * n,
                6.0 * t * dm * di + 6.0 * t * di * n)

    def experts(t, dm, f, ex, k):
        return (t * (2 * dm * e + 8 * ex + 4 * k) + min(ex, t * k) * dm * f / 2.0,
                4.0 * t * k * dm * f)

    if kind == "moe":
        b, f = experts(case["rows"], case["d_model"], case["d_ff"], case["experts"],
                       case["top_k"])
        return {"bytes": b, "flops": f}
    if kind in ("layer", "block"):
        t, dm = int(_offsets(case)[-1]), case["d_model"]
        b, f = mamba(t, case["seqs"], dm, case["d_state"])
        if kind == "block":
            b2, f2 = experts(t, dm, 4 * dm, case["experts"], case["top_k"])
            # the experts' input and the Mamba core's output stay inside the block
            b, f = b + b2 - t * dm * e, f + f2
        return {"bytes": b, "flops": f}
    dm, n, inner = case["d_model"], case["d_state"], 64 * case["heads"]
    t = int(_offsets(case)[-1]) if kind == "mamba2" else case["rows"]
    small = 2 * n + case["heads"]
    flops = t * (6.0 * dm * inner + 2.0 * dm * small + 6.0 * inner * n)
    weights = 3 * dm * inner / 4 + 4.0 * dm * small
    if kind == "mamba2":
        return {"bytes": 2 * t * dm * e + weights + 4.0 * case["seqs"] * inner * n, "flops": flops}
    return {"bytes": 2 * t * dm * e + weights + 8.0 * t * (inner * n + 3 * (inner + 2 * n)),
            "flops": flops}


def tolerance(case):
    """Measured as the difference from exact() and between summation orders.  A last-bit change
    before a quantization moves an int8 code by one in a few of 10^4 places (1 part in 127 of the
    row's largest value), which is what the paths with a scan before a projection show; bf16
    storage rounds at 2^-9."""
    kind = case["kind"]
    if kind == "linear":
        return {"rel": 1e-5, "max": 1e-4} if case["dtype"] == "f32" else {"rel": 4e-3, "max": 2e-2}
    if kind == "train":
        return {"rel": 1e-5, "max": 1e-4}
    if kind == "scan_step":
        return {"rel": 2e-5, "max": 1e-3} if case["dtype"] == "f32" else {"rel": 5e-3, "max": 2e-2}
    if case["dtype"] == "f32":
        return {"rel": 3e-3, "max": 0.1}
    return {"rel": 1e-2, "max": 0.2}


# ---- the same in 64 bits ----------------------------------------------------------

def _ternary(w):
    """Packed weights in float64: absmean codes in {-1, 0, +1} times the weight scale."""
    scale = w.double().abs().mean().item()
    scale = float(np.float32(np.float32(scale) + np.float32(1e-8)))
    denom = float(np.float32(np.float32(scale) + np.float32(1e-8)))
    v = w.double() / denom
    return ((v > 0.5).double() - (v < -0.5).double()), scale


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _codes(x, rms):
    """int8 codes and scale of float64 rows (per-row absmax, round half to even)."""
    x = _rms(x, 1e-6) if rms else x
    m = x.abs().amax(-1, keepdim=True) + 1e-8
    return torch.clamp(torch.round(x * (127.0 / m)), -127, 127), m / 127.0


def _bitlinear(x, w, rms=True):
    q, s = _codes(x, rms)
    t, ws = _ternary(w)
    return (q @ t.t()) * (s * ws)


def _silu(v):
    return v * torch.sigmoid(v)


def _conv(x, w, b, cu):
    """Causal depthwise convolution + bias + SiLU per sequence, x [T, C] float64."""
    out = torch.empty_like(x)
    taps = w.shape[1]
    for a, e in zip(cu[:-1].tolist(), cu[1:].tolist()):
        seg = torch.cat([x.new_zeros(taps - 1, x.shape[1]), x[a:e]])
        acc = sum(seg[j:j + e - a] * w[:, j].double() for j in range(taps))
        out[a:e] = _silu(acc + b.double())
    return out


def _scan(x, delta, a, B, C, skip, cu):
    """The selective scan of float64 rows: x [T, C], delta [T, C], a [C, N] (or [C, 1], one decay
    per channel), B, C [T, N] -> y [T, C], final states [S, C, N].  The sequences step together,
    longest first, so that the running ones are always the first."""
    lengths = cu[1:] - cu[:-1]
    order = np.argsort(-lengths, kind="stable")
    start = torch.from_numpy(cu[:-1][order].astype(np.int64)).to(x.device)
    lens = lengths[order]
    state = x.new_zeros(len(order), x.shape[1], B.shape[1])
    y = torch.empty_like(x)
    for t in range(int(lens[0])):
        live = int((lens > t).sum())
        row = start[:live] + t
        dl, xr = delta[row], x[row]
        st = state[:live]
        st.mul_(torch.exp(dl[:, :, None] * a)).add_((dl * xr)[:, :, None] * B[row][:, None, :])
        y[row] = torch.matmul(st, C[row][:, :, None])[:, :, 0] + skip * xr
    final = torch.empty_like(state)
    final[torch.from_numpy(order.copy()).to(x.device)] = state
    return y, final


def _softplus(v):
    return torch.nn.functional.softplus(v, threshold=1e9)


def _mamba_layer(d, h):
    di = d["d_skip"].shape[0]
    xz = _bitlinear(h, d["w_in"])
    x = _conv(xz[:, :di], d["conv_w"], d["conv_b"], d["cu"])
    y, final = _scan(x, _softplus(d["dt"].double()), -torch.exp(d["a_log"].double()),
                     d["B"].double(), d["C"].double(), d["d_skip"].double(), d["cu"])
    y *= _silu(xz[:, di:])
    return _bitlinear(y, d["w_out"]), final


def _experts(d, x, k):
    p = torch.softmax(d["logits"].double(), -1)
    top, sel = torch.topk(p, k, dim=-1)
    if k < p.shape[1]:
        top = top / top.sum(-1, keepdim=True)
    weights = torch.zeros_like(p).scatter_(1, sel, top)
    out = torch.zeros_like(x)
    for e in range(p.shape[1]):
        rows = torch.nonzero(weights[:, e])[:, 0]
        if rows.numel():
            h = torch.relu(_bitlinear(x[rows], d["w_up"][e])) ** 2
            out[rows] += weights[rows, e, None] * _bitlinear(h, d["w_down"][e])
    return out, weights


def _mamba2_head(d):
    u = d["u"].double()
    xv, z = _bitlinear(u, d["w_x"], False), _bitlinear(u, d["w_z"], False)
    f = [u @ d[k].double().t() for k in ("w_B", "w_C", "w_dt")]
    return xv, z, f[0], f[1], _softplus(f[2] + d["dt_bias"].double())


def _mamba2_tail(d, y, z):
    return _bitlinear(_rms(y * _silu(z), 1e-5) * d["norm_w"].double(), d["w_out"], False)


def exact(case, seed):
    kind = case["kind"]
    d = _data(case, seed)
    if kind == "linear":
        y = _bitlinear(d["x"].double(), d["w"])
        return y if d["mag"] is None else y * d["mag"].double() + d["bias"].double()
    if kind == "layer":
        out, final = _mamba_layer(d, d["x"].double())
        return {"out": out, "final_state": final}
    if kind == "block":
        x = d["x"].double()
        core, final = _mamba_layer(d, _rms(x, 1e-6) * d["core_gamma"].double())
        r = x + core
        ff, _ = _experts(d, _rms(r, 1e-6) * d["ff_gamma"].double(), case["top_k"])
        return {"out": r + ff, "residual": r, "final_state": final}
    if kind == "moe":
        out, weights = _experts(d, d["x"].double(), case["top_k"])
        return {"out": out, "weights": weights, "selected": None}
    if kind == "scan_step":
        x, delta = d["x"].double(), _softplus(d["dt"].double())
        st = d["state"].double() * torch.exp(delta[:, :, None] * -torch.exp(d["a_log"].double()))
        st += (delta * x)[:, :, None] * d["B"].double()[:, None, :]
        y = torch.matmul(st, d["C"].double()[:, :, None])[:, :, 0] + d["D"].double() * x
        return {"y": y * _silu(d["z"].double()), "state": st}
    if kind in ("mamba2", "mamba2_step"):
        xv, z, B, C, delta = _mamba2_head(d)
        inner, n = xv.shape[1], B.shape[1]
        per = lambda v: v.repeat_interleave(64, -1)
        a, skip = -torch.exp(per(d["a_log"].double())), per(d["d_skip"].double())
        if kind == "mamba2":
            xbc = _conv(torch.cat([xv, B, C], 1), d["conv_w"], d["conv_b"], d["cu"])
            y, final = _scan(xbc[:, :inner], per(delta), a[:, None], xbc[:, inner:inner + n],
                             xbc[:, inner + n:], skip, d["cu"])
            return {"out": _mamba2_tail(d, y, z), "final_state": final}
        raw = torch.cat([xv, B, C], 1)
        win = torch.cat([d["ring"].double(), raw[:, None]], 1)
        xbc = _silu((win * d["conv_w"].double().t()).sum(1) + d["conv_b"].double())
        x, B, C, delta = xbc[:, :inner], xbc[:, inner:inner + n], xbc[:, inner + n:], per(delta)
        st = d["state"].double() * torch.exp(delta * a)[:, :, None]
        st += (delta * x)[:, :, None] * B[:, None, :]
        y = torch.matmul(st, C[:, :, None])[:, :, 0] + skip * x
        return {"out": _mamba2_tail(d, y, z), "state": st, "ring": win[:, 1:]}
    x, grad = d["x"].double(), d["grad"].double()
    q, s = _codes(x, case["rms"])
    t, ws = _ternary(d["w"])
    pre = (q @ t.t()) * (s * ws)
    y, gp, got = pre, grad, {}
    if d["mag"] is not None:
        y, gp = pre * d["mag"].double() + d["bias"].double(), grad * d["mag"].double()
        got.update(dmag=(grad * pre).sum(0), dbias=grad.sum(0))
    keep = (d["w"].double() / float(np.float32(ws + 1e-8))).abs() <= 1.0
    dw = (gp.t() @ (q * s)) * keep
    dx = gp @ (t * ws)
    if case["rms"]:
        inv = 1.0 / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6)
        xn = x * inv
        dx = (dx - xn * (dx * xn).mean(-1, keepdim=True)) * inv
    return {"y": y, "dx": dx, "dW": dw, **got}
