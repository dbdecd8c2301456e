"""Batches on the pair GEMM: column-major Q4_0 at many tokens and fp16
weights whose rows are no multiple of 64, at the edges of its tiles (row tiles
of 32 and 64 tokens, 256 output columns, 64-column stages cut in half), with
short buffers, scales past fp16's products, infinities and biases.
(test_routes.py checks which kernel each case runs.)"""
import ctypes

import numpy as np
import pytest


def _p(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def _col_f64(orc, wb, x, bias, n, m):
    return np.stack([orc.matmul_q4_0_col_f64(wb, r, bias, n, m) for r in x])


def _col(torch, wb, x, bias, n, m):
    from hypno_amd import _lib
    dw, dx = torch.from_numpy(wb).cuda(), torch.from_numpy(x).cuda()
    db = torch.from_numpy(bias).cuda() if bias is not None else None
    y = torch.full((x.shape[0], n), float("nan"), device="cuda")
    st = _lib.load().hypno_hip_matmul_q4_0_col_dev(_p(y), _p(dw), wb.size, _p(dx), _p(db), n, m,
                                                   x.shape[0], None)
    assert st == 0
    torch.cuda.synchronize()
    return y.cpu().numpy()


COL_CASES = [  # tokens, n, m, bytes cut off the end
    (40, 2080, 2080, 0), (33, 3104, 1056, 0), (65, 1056, 1120, 0), (128, 256, 2048, 0),
    (300, 544, 1056, 0), (64, 1056, 1056, 18 * 33 * 100 + 7), (8, 5664, 2080, 0),
    (300, 14336, 544, 18 * 448 * 3),
    # 64-row tiles, one and several K pieces
    (100, 16480, 96, 0), (35, 11584, 928, 0), (100, 5632, 1056, 18 * 176 * 20),
    # an odd number of blocks that ends the buffer: one token at a time
    (129, 1024, 1024, 18)]


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,n,m,cut", COL_CASES)
def test_col_major_many_tokens(orc, tokens, n, m, cut):
    import torch
    print(f"col tokens={tokens} n={n} m={m} cut={cut}", flush=True)
    rng = np.random.default_rng(tokens + n)
    wb = orc.quantize_q4_0((rng.standard_normal(n * m) * 0.02).astype(np.float32))
    wb = np.ascontiguousarray(wb[:wb.size - cut])
    x = rng.standard_normal((tokens, m)).astype(np.float32)
    x[:, ::61] *= 20.0
    bias = rng.standard_normal(n).astype(np.float32)
    got = _col(torch, wb, x, bias, n, m)
    ref = _col_f64(orc, wb, x, bias, n, m)
    # fp32 sums of exact products: random error well under sqrt(K) 2^-24
    for t in range(tokens):
        assert orc.normwise_err(got[t], ref[t]) <= 2e-5, t


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,n,m", [(40, 2080, 2080), (35, 11584, 928)])
@pytest.mark.parametrize("bits", [0x6FFF, 0x7000, 0x7BFF, 0x0001, 0x8200])
def test_col_major_scale_range(orc, bits, tokens, n, m):
    """One block's scale at the largest whose products fp16 holds, past it, at
    fp16's largest value, at its smallest and at a negative subnormal, on 32- and
    64-row tiles."""
    import torch
    rng = np.random.default_rng(bits)
    wb = orc.quantize_q4_0((rng.standard_normal(n * m) * 0.02).astype(np.float32))
    g = 777 * (n // 32) + 13
    wb[18 * g:18 * g + 2] = np.frombuffer(np.uint16(bits).tobytes(), np.uint8)
    x = rng.standard_normal((tokens, m)).astype(np.float32)
    got = _col(torch, wb, x, None, n, m)
    ref = _col_f64(orc, wb, x, None, n, m)
    for t in range(tokens):
        assert orc.normwise_err(got[t], ref[t]) <= 2e-5, t
    # the other block columns on their own
    keep = np.r_[0:13 * 32, 14 * 32:n]
    for t in range(tokens):
        assert orc.normwise_err(got[t][keep], ref[t][keep]) <= 2e-5, t


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,n,m", [(40, 2080, 2080), (35, 11584, 928)])
def test_col_major_infinite_token(orc, tokens, n, m):
    import torch
    rng = np.random.default_rng(3)
    wb = orc.quantize_q4_0((rng.standard_normal(n * m) * 0.02).astype(np.float32))
    x = rng.standard_normal((tokens, m)).astype(np.float32)
    x[7, 100] = np.inf
    got = _col(torch, wb, x, None, n, m)
    w = orc.dequantize_q4_0(wb).reshape(m, n)[100]
    want = np.full(n, np.nan)
    want[w != 0] = np.sign(w[w != 0]) * np.inf
    assert np.array_equal(got[7], want.astype(np.float32), equal_nan=True)
    ref = _col_f64(orc, wb, x[8:], None, n, m)
    for t in range(8, tokens):
        assert orc.normwise_err(got[t], ref[t - 8]) <= 2e-5, t


F16_CASES = [(2, 20001, 1056), (3, 20001, 1056), (16, 2600, 992), (33, 1300, 1120),
             (65, 257, 2400), (129, 511, 1056), (300, 300, 544), (70, 16384, 1056),
             (100, 16480, 96), (35, 11590, 928)]  # the last two: 64-row tiles


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,n,m", F16_CASES)
def test_f16_half_stage_rows(orc, tokens, n, m):
    import torch

    import hypno_amd as hk
    print(f"f16 tokens={tokens} n={n} m={m}", flush=True)
    rng = np.random.default_rng(tokens + n)
    w = (rng.standard_normal(n * m) * 0.02).astype(np.float16)
    x = rng.standard_normal((tokens, m)).astype(np.float32)
    dw = torch.from_numpy(w.view(np.uint8)).cuda()
    dx = torch.from_numpy(x).cuda()
    y = torch.full((tokens, n), float("nan"), device="cuda")
    hk.batch_matmul(y, dw, hk.DType.FP16, dx, n, m, tokens)
    torch.cuda.synchronize()
    got = y.cpu().numpy()
    ref = x.astype(np.float64) @ w.reshape(n, m).astype(np.float64).T
    for t in range(tokens):
        assert orc.normwise_err(got[t], ref[t]) <= 2e-5, t


def _outliers(rng, tokens, m, k):
    """Ordinary tokens, and the same with values 2^12 to 2^100 at column k."""
    x = rng.standard_normal((tokens, m)).astype(np.float32)
    big = x.copy()
    big[:, k] = np.ldexp(np.float32(1.0), 12 + np.arange(tokens) * 88 // (tokens - 1))
    x[:, k] = 0.0
    return x, big


# Exact products; the random rounding of their fp32 sums stays under 4 2^-24 of
# the result's norm (measured: 1 to 2 2^-24).
OUTLIER_TOL = 4 * 2.0 ** -24


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,n,m", [(128, 5632, 2048), (16, 2048, 2080)])
def test_col_major_outlier(orc, tokens, n, m):
    """Tokens whose largest value meets weights of zero: outputs are as accurate
    as if that input were not there."""
    import torch
    print(f"col tokens={tokens} n={n} m={m}", flush=True)
    rng = np.random.default_rng(n)
    w = (rng.standard_normal((m, n)) * 0.02).astype(np.float32)
    w[100] = 0.0
    wb = orc.quantize_q4_0(w.ravel())
    x, big = _outliers(rng, tokens, m, 100)
    got = _col(torch, wb, big, None, n, m)
    ref = _col_f64(orc, wb, x, None, n, m)
    for t in range(tokens):
        assert orc.rel_l2(got[t], ref[t]) <= OUTLIER_TOL, t


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,n,m", [(200, 7200, 2848), (8, 4096, 2080)])
def test_f16_outlier(orc, tokens, n, m):
    import torch

    import hypno_amd as hk
    print(f"f16 tokens={tokens} n={n} m={m}", flush=True)
    rng = np.random.default_rng(n)
    w = (rng.standard_normal((n, m)) * 0.02).astype(np.float16)
    w[:, 100] = 0.0
    x, big = _outliers(rng, tokens, m, 100)
    y = torch.full((tokens, n), float("nan"), device="cuda")
    hk.batch_matmul(y, torch.from_numpy(w.view(np.uint8)).cuda(), hk.DType.FP16,
                    torch.from_numpy(big).cuda(), n, m, tokens)
    torch.cuda.synchronize()
    got, ref = y.cpu().numpy(), x.astype(np.float64) @ w.astype(np.float64).T
    for t in range(tokens):
        assert orc.rel_l2(got[t], ref[t]) <= OUTLIER_TOL, t
