"""Tokens that hold infinities, NaN or values near fp32's largest, on the kernels
for rows outside the tuned kernels' stages.  A token with one infinity has +-inf
where that column's weight is not zero and NaN where it is, whatever finite
values stand beside it; other tokens keep their fp32 accuracy."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _run(torch, fn, wb, x, n, m):
    from hypno_amd import _lib
    dw, dx = torch.from_numpy(wb).cuda(), torch.from_numpy(x).cuda()
    y = torch.full((x.shape[0], n), float("nan"), device="cuda")
    st = getattr(_lib.load(), fn)(_p(y), _p(dw), wb.size, _p(dx), None, n, m, x.shape[0], None)
    assert st == 0
    torch.cuda.synchronize()
    return y.cpu().numpy()


def _tokens(rng, tokens, m):
    """Ordinary tokens, and four with special values (tokens 1 to 4)."""
    x = rng.standard_normal((tokens, m)).astype(np.float32)
    x[1, 100] = np.inf
    x[1, 101:140:2], x[1, 102:140:2] = 1e5, -1e5     # past fp16's range
    x[2, 7] = -np.inf
    x[2, 8:40:2], x[2, 9:40:2] = 3e38, -3e38
    x[3, 50] = np.nan
    x[4, 20] = 3.3e38                                # finite, near the largest
    return x


def _check(orc, got, x, w):
    """w: the exact weights [n][m] in float64."""
    for t, k in ((1, 100), (2, 7)):
        with np.errstate(invalid="ignore"):
            want = np.sign(w[:, k]) * x[t, k]  # 0 * inf: NaN
        assert np.array_equal(got[t], want.astype(np.float32), equal_nan=True), t
    assert np.isnan(got[3]).all()
    # fp32 sums: random error under sqrt(K) 2^-24 of the largest output
    for t in [0, *range(4, x.shape[0])]:
        assert orc.normwise_err(got[t], x[t].astype(np.float64) @ w.T) <= 2e-5, t


@pytest.mark.parametrize("dt", ["q4_0", "q8_0"])
@pytest.mark.parametrize("tokens,n,m", [(17, 2400, 2080), (9, 7200, 2144)])
def test_block_batch(orc, dt, tokens, n, m):
    import torch
    print(f"{dt} tokens={tokens} n={n} m={m}", flush=True)
    rng = np.random.default_rng(n)
    f = (rng.standard_normal(n * m) * 0.02).astype(np.float32)
    wb = orc.quantize_q4_0(f) if dt == "q4_0" else orc.quantize_q8_0(f)
    w = (orc.dequantize_q4_0 if dt == "q4_0" else orc.dequantize_q8_0)(wb)
    x = _tokens(rng, tokens, m)
    got = _run(torch, f"hypno_hip_matmul_{dt}_dev", wb, x, n, m)
    _check(orc, got, x, w[:n * m].reshape(n, m).astype(np.float64))


@pytest.mark.parametrize("tokens,n,m", [(8, 300, 1056), (70, 520, 2080)])
def test_f16_batch(orc, tokens, n, m):
    """fp16 rows of K % 64 == 32, finite and with infinite weights in columns
    where tokens hold values that fp16 has exactly (a zero lo part) and not."""
    import torch
    print(f"f16 tokens={tokens} n={n} m={m}", flush=True)
    rng = np.random.default_rng(n + m)
    w = (rng.standard_normal((n, m)) * 0.02).astype(np.float16)
    x = _tokens(rng, tokens, m)
    x[5, 33], x[6, 33], x[7, 33] = 1.0, -2.5, 0.0
    fn = "hypno_hip_matmul_f16_dev"
    _check(orc, _run(torch, fn, w.ravel().view(np.uint8), x, n, m), x, w.astype(np.float64))
    inf = {3: (33, np.inf), n // 2: (33, -np.inf), n - 1: (m - 1, np.inf)}
    for r, (k, v) in inf.items():
        w[r, k] = v
    got = _run(torch, fn, w.ravel().view(np.uint8), x, n, m)
    one = np.concatenate([_run(torch, fn, w.ravel().view(np.uint8), x[t:t + 1], n, m)
                          for t in range(tokens)])  # the one-token product: fp32 FMAs
    for r in inf:
        assert np.array_equal(got[:, r], one[:, r], equal_nan=True), r
    rest = np.setdiff1d(np.arange(n), list(inf))
    _check(orc, got[:, rest], x, w[rest].astype(np.float64))


@pytest.mark.parametrize("dt", ["q4_0", "q8_0"])
@pytest.mark.parametrize("n,m", [(33, 96), (300, 544), (257, 2080)])
def test_one_token_near_the_largest(orc, dt, n, m):
    """One token whose values times the blocks' integers leave fp32, times the
    weights not."""
    import torch
    print(f"{dt} n={n} m={m}", flush=True)
    rng = np.random.default_rng(n)
    f = (rng.standard_normal(n * m) * 0.02).astype(np.float32)
    wb = orc.quantize_q4_0(f) if dt == "q4_0" else orc.quantize_q8_0(f)
    w = (orc.dequantize_q4_0 if dt == "q4_0" else orc.dequantize_q8_0)(wb)
    w = w[:n * m].reshape(n, m).astype(np.float64)
    x = rng.standard_normal((1, m)).astype(np.float32)
    x[0, 3:40:3] = np.float32(3e38) * np.sign(x[0, 3:40:3])
    got = _run(torch, f"hypno_hip_matmul_{dt}_dev", wb, x, n, m)
    assert orc.normwise_err(got[0], x[0].astype(np.float64) @ w.T) <= 2e-5
    x[0, 3] = np.inf
    got = _run(torch, f"hypno_hip_matmul_{dt}_dev", wb, x, n, m)
    with np.errstate(invalid="ignore"):
        want = w[:, 3] * np.inf
    assert np.array_equal(got[0], want.astype(np.float32), equal_nan=True)
