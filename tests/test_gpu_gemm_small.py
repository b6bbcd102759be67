"""The small-tile ternary GEMMs (32 / 64 outputs x 32 / 64 tokens, K split over four waves) at the
edges of their tiles and of the rule that picks them, on both weight layouts: accumulators and
outputs bit for bit against the integer product and the reference's affine (each step rounded)."""
import numpy as np
import pytest
import torch

from reimagined_amd import ops

pytestmark = pytest.mark.gpu


def _matrix(rng, n, k):
    codes = rng.integers(-1, 2, (n, k)).astype(np.int64)
    words = ((codes + 1).astype(np.uint32).reshape(n * k // 16, 16) << (2 * np.arange(16, dtype=np.uint32)))
    return codes, words.sum(1, dtype=np.uint32)


def _affine(acc, s, ws, mag, bias):
    v = acc.astype(np.float32) * (s * np.float32(ws))[:, None]
    if mag is not None:
        v = v * mag
    return v if bias is None else v + bias


# K of 1, 2, 3, 4, 5 and 9 blocks of 128 (waves with no block, uneven quarters); row counts and
# widths on either side of 32 / 64; 3001 rows, the most that the 64 x 64 tiles take here
@pytest.mark.parametrize("m,k,n", [(2, 128, 32), (9, 256, 33), (31, 384, 7), (32, 512, 64),
                                   (33, 640, 100), (64, 1152, 129), (65, 128, 768), (100, 2048, 8192),
                                   (300, 768, 768), (257, 1024, 4104), (700, 2048, 1000),
                                   (3001, 2048, 520)])
@pytest.mark.parametrize("mfma", [True, False])
@pytest.mark.parametrize("ydt", [torch.float32, torch.bfloat16])
def test_small_tiles_bit_exact(dev, m, k, n, mfma, ydt):
    rng = np.random.default_rng(m + 3 * k + n)
    codes, words = _matrix(rng, n, k)
    q = rng.integers(-127, 128, (m, k)).astype(np.int8)
    s = rng.uniform(0.01, 0.1, m).astype(np.float32)
    mag = rng.uniform(0.5, 1.5, n).astype(np.float32) if n % 2 == 0 else None
    bias = rng.standard_normal(n).astype(np.float32) if m % 2 == 0 else None
    t = lambda a: None if a is None else torch.from_numpy(a).to(dev)
    packed = t(words.view(np.int32))
    if mfma:
        y, acc = ops.ternary_gemm_mfma(t(q), t(s), ops.pack_mfma_layout(packed), 0.37, n, t(mag),
                                       t(bias), out_dtype=ydt, want_acc=True)
    else:
        y, acc = ops.ternary_gemm(t(q), t(s), packed, 0.37, n, t(mag), t(bias), out_dtype=ydt,
                                  want_acc=True, path=1)
    # |acc| <= 127 * 2048: exact in float64
    want = np.rint(q.astype(np.float64) @ codes.T.astype(np.float64)).astype(np.int32)
    np.testing.assert_array_equal(acc.cpu().numpy(), want)
    wy = torch.from_numpy(_affine(want, s, 0.37, mag, bias)).to(ydt)
    np.testing.assert_array_equal(y.float().cpu().numpy(), wy.float().numpy())


@pytest.mark.parametrize("rows", [[5], [0, 1, 33, 64, 65, 0, 31, 2], [12] * 8, [0, 0, 200, 0],
                                  [130, 7, 64, 300]])
@pytest.mark.parametrize("k,n", [(128, 96), (1024, 520), (4096, 256)])
@pytest.mark.parametrize("gather", [True, False])
def test_grouped_small_tiles_bit_exact(dev, rows, k, n, gather):
    rng = np.random.default_rng(sum(rows) + k + n)
    slots = sum(rows)
    mats = [_matrix(rng, n, k) for _ in rows]
    mags = [rng.uniform(0.5, 1.5, n).astype(np.float32) for _ in rows]
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    views = ops.LinearViewArray([(ops.pack_mfma_layout(t(w.view(np.int32))), 0.3 + 0.01 * e, k, n,
                                  t(mags[e]) if e % 2 else None, None)
                                 for e, (_, w) in enumerate(mats)], dev)
    offsets = np.concatenate([[0], np.cumsum(rows)]).astype(np.int32)
    perm = rng.permutation(slots).astype(np.int32)
    q = rng.integers(-127, 128, (slots, k)).astype(np.int8)
    s = rng.uniform(0.01, 0.1, slots).astype(np.float32)
    ws = torch.empty(ops.grouped_mfma_workspace_bytes(), dtype=torch.uint8, device=dev)
    for sq, work in ((False, None), (True, ws)):
        y = ops.grouped_ternary_gemm_mfma(views, t(offsets), t(perm), t(q), t(s), n, slots,
                                          squared_relu=sq, gather=gather, workspace=work)
        want = np.empty((slots, n), np.float32)
        for e, (codes, _) in enumerate(mats):
            seg = np.arange(offsets[e], offsets[e + 1])
            src = perm[seg] if gather else seg
            acc = np.rint(q[src].astype(np.float64) @ codes.T.astype(np.float64))
            v = _affine(acc, s[src], np.float32(0.3 + 0.01 * e), mags[e] if e % 2 else None, None)
            if sq:
                v = np.where(v > 0, v, np.float32(0))
                v = v * v
            want[seg] = v
        np.testing.assert_array_equal(y.cpu().numpy(), want)


# The last row counts of the small tiles and the first of the 256 x 128 ones at one width (by the
# rule 143 against 174 tenths of a us, then 192 against 174)
@pytest.mark.parametrize("m", [200, 300])
@pytest.mark.parametrize("mfma", [True, False])
def test_either_side_of_the_rule_bit_exact(dev, m, mfma):
    test_small_tiles_bit_exact(dev, m, 2048, 8192, mfma, torch.float32)


# 64 x 64 tiles per expert (rows around a multiple of 64, an expert without rows, a width that is
# not one), which the cases above never pick
@pytest.mark.parametrize("k,n", [(1024, 2000), (2048, 1000)])
@pytest.mark.parametrize("gather", [True, False])
def test_grouped_64_by_64_tiles_bit_exact(dev, k, n, gather):
    test_grouped_small_tiles_bit_exact(dev, [200, 130, 64, 0, 65, 241], k, n, gather)


# Either side of the rule that keeps few rows of a long K on the GEMV
@pytest.mark.parametrize("m,k,n", [(2, 2048, 68), (2, 2176, 68), (2, 2176, 8192), (2, 2176, 8196),
                                   (2, 8192, 8196), (3, 8064, 36), (4, 8192, 2048), (4, 8192, 2052),
                                   (5, 8192, 68)])
def test_few_rows_of_long_k_bit_exact(dev, m, k, n):
    rng = np.random.default_rng(m + k + n)
    codes, words = _matrix(rng, n, k)
    q = rng.integers(-127, 128, (m, k)).astype(np.int8)
    s = rng.uniform(0.01, 0.1, m).astype(np.float32)
    t = lambda a: torch.from_numpy(a).to(dev)
    y, acc = ops.ternary_gemm(t(q), t(s), t(words.view(np.int32)), 0.37, n, want_acc=True)
    want = np.rint(q.astype(np.float64) @ codes.T.astype(np.float64)).astype(np.int32)
    np.testing.assert_array_equal(acc.cpu().numpy(), want)
    np.testing.assert_array_equal(y.cpu().numpy(), _affine(want, s, 0.37, None, None))


# More experts than a wave has lanes, most of them without rows: the first, the last, at a multiple
# of 64 and past it
@pytest.mark.parametrize("rows", [{0: 1, 1: 33}, {63: 40, 64: 2, 69: 31}, {127: 5, 128: 70, 129: 1},
                                  {e: e % 3 for e in range(130)}])
@pytest.mark.parametrize("gather", [True, False])
def test_grouped_many_experts_bit_exact(dev, rows, gather):
    test_grouped_small_tiles_bit_exact(dev, [rows.get(e, 0) for e in range(130)], 128, 96, gather)
