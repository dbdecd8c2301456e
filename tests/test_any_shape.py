"""Q4_0 and Q8_0 products at row lengths that no tuned kernel takes: one token
through the any-length GEMV, batches through the fp32-accurate block GEMM (and,
for Q4_0 from 16 tokens at K % 64 == 0, the prefill GEMM).  The cases sit at
the edges of their tiles: odd numbers of blocks per row (rows on 2-byte
boundaries), buffers that end with the last row, x off a 16-byte boundary, one
row or column past a tile, K pieces, lanes shared by several short rows.  (test_routes.py checks which kernel
each case runs.)"""
import ctypes

import numpy as np
import pytest

CASES = [  # dtype, tokens, n, m
    (dt, tok, n, m)
    for dt in ("q4_0", "q8_0")
    for tok, n, m in [
        # the any-length GEMV: 8, 16, 32 and 64 lanes per row
        (1, 1, 32), (1, 33, 96), (1, 257, 288), (1, 31, 544), (1, 100, 1056), (1, 65, 11008),
        (1, 7, 32768), (1, 5, 32800), (2, 97, 1120), (7, 513, 4128), (33, 257, 2080),
        # too few products or a buffer that ends inside a dword: token by token
        (5, 4097, 4128), (300, 257, 1120),
        # the block GEMM, odd numbers of blocks per row, 32-row tiles, a row or column
        # past them, one and several K pieces
        (16, 1300, 4128), (33, 1030, 2400), (64, 520, 2464), (65, 1290, 1120),
        (129, 600, 1120), (129, 8194, 96),
        # 64-row tiles, one and several K pieces
        (100, 16480, 96), (33, 11086, 736),
        # whole 64-column stages: the block GEMM on even numbers of blocks below 16
        # tokens, from 16 the prefill GEMMs
        (8, 7200, 1472), (15, 4162, 1344), (2, 16000, 2880), (15, 33000, 192), (16, 640, 2880),
        (17, 129, 4160)]
]


def _run(lib, torch, dt, wb, x, bias, n, m, tokens, shift):
    buf = torch.empty(x.size + shift, dtype=torch.float32, device="cuda")
    dx = buf[shift:]
    dx.copy_(torch.from_numpy(x.ravel()))
    dw = torch.from_numpy(wb).cuda()
    db = torch.from_numpy(bias).cuda()
    y = torch.full((tokens * n,), float("nan"), dtype=torch.float32, device="cuda")
    fn = {"q4_0": lib.hypno_hip_matmul_q4_0_dev, "q8_0": lib.hypno_hip_matmul_q8_0_dev}[dt]
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    assert fn(p(y), p(dw), wb.size, p(dx), p(db), n, m, tokens, None) == 0
    torch.cuda.synchronize()
    return y.cpu().numpy().reshape(tokens, n)


@pytest.mark.gpu
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("dt,tokens,n,m", CASES)
def test_any_shape(orc, dt, tokens, n, m, shift):
    import torch

    from hypno_amd import _lib
    print(f"{dt} tokens={tokens} n={n} m={m} shift={shift}", flush=True)
    rng = np.random.default_rng(n * 7 + m + tokens)
    w = (rng.standard_normal(n * m) * 0.02).astype(np.float32)
    wb = orc.quantize_q4_0(w) if dt == "q4_0" else orc.quantize_q8_0(w)
    x = rng.standard_normal((tokens, m)).astype(np.float32)
    x[:, ::97] *= 30.0
    bias = rng.standard_normal(n).astype(np.float32)
    got = _run(_lib.load(), torch, dt, wb, x, bias, n, m, tokens, shift)
    f64 = orc.matmul_q4_0_f64 if dt == "q4_0" else orc.matmul_q8_0_f64
    ref = np.stack([f64(wb, x[t], bias, n, m) for t in range(tokens)])
    # from 16 tokens whole 64-column stages round x to fp16 (relative 2^-12 at
    # random, 3e-4 of the result at most here); everything else is fp32 sums,
    # whose random error stays under sqrt(K) 2^-24 of the largest product sum
    if tokens >= 16 and m % 64 == 0:
        assert orc.rel_l2(got, ref) <= 2e-3
    else:
        for t in range(tokens):
            assert orc.normwise_err(got[t], ref[t]) <= 2e-5, t


@pytest.mark.gpu
def test_any_shape_plan_and_capture(orc):
    """A plan's job with K = 11008 (any-length GEMV), and a ragged batch
    captured on a stream that has no workspace yet, replayed."""
    import torch

    import hypno_amd as hk
    n, m, tokens = 320, 1120, 24
    rng = np.random.default_rng(5)
    wb = orc.quantize_q4_0((rng.standard_normal(n * 11008) * 0.02).astype(np.float32))
    x = rng.standard_normal(11008).astype(np.float32)
    dw, dx = torch.from_numpy(wb).cuda(), torch.from_numpy(x).cuda()
    y = torch.full((n,), float("nan"), device="cuda")
    plan = hk.GemvPlan([(y, dw, dx, None, n, 11008)])
    plan.run()
    torch.cuda.synchronize()
    assert orc.normwise_err(y.cpu().numpy(), orc.matmul_q4_0_f64(wb, x, None, n, 11008)) <= 2e-5
    wb = orc.quantize_q4_0((rng.standard_normal(n * m) * 0.02).astype(np.float32))
    xb = rng.standard_normal((tokens, m)).astype(np.float32)
    dw, dx = torch.from_numpy(wb).cuda(), torch.from_numpy(xb).cuda()
    y = torch.zeros(tokens, n, device="cuda")
    ref = np.stack([orc.matmul_q4_0_f64(wb, xb[t], None, n, m) for t in range(tokens)])
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        hk.batch_matmul(y, dw, hk.DType.Q4_0, dx, n, m, tokens)
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        for t in range(tokens):
            assert orc.normwise_err(y[t].cpu().numpy(), ref[t]) <= 2e-5


@pytest.mark.gpu
@pytest.mark.parametrize("dt", ["q4_0", "q8_0"])
@pytest.mark.parametrize("tokens,n,m", [(8, 7200, 1440), (40, 1100, 2080), (70, 1300, 2080)])
def test_any_shape_outlier(orc, dt, tokens, n, m):
    """Tokens whose largest values, 2^12 to 2^100 times the others, stand in
    columns of zero weights: outputs keep the accuracy of fp32 sums, as if
    those columns were not there."""
    import torch

    from hypno_amd import _lib
    print(f"{dt} tokens={tokens} n={n} m={m}", flush=True)
    rng = np.random.default_rng(n)
    w = (rng.standard_normal((n, m)) * 0.02).astype(np.float32)
    w[:, 96:128] = 0.0  # one block
    wb = (orc.quantize_q4_0 if dt == "q4_0" else orc.quantize_q8_0)(w.ravel())
    x = rng.standard_normal((tokens, m)).astype(np.float32)
    small = x.copy()
    x[:, 100] = np.ldexp(np.float32(1.0), 12 + np.arange(tokens) * 88 // max(tokens - 1, 1))
    small[:, 96:128] = 0.0
    bias = np.zeros(n, np.float32)
    got = _run(_lib.load(), torch, dt, wb, x, bias, n, m, tokens, 0)
    ref = np.stack([(orc.matmul_q4_0_f64 if dt == "q4_0" else orc.matmul_q8_0_f64)(
        wb, small[t], bias, n, m) for t in range(tokens)])
    # exact products; random rounding of K / 32 block sums and the 32 products of
    # each stays under 8 2^-24 of the result's norm (measured: about 4 2^-24)
    for t in range(tokens):
        assert orc.rel_l2(got[t], ref[t]) <= 8 * 2.0 ** -24, t


@pytest.mark.gpu
@pytest.mark.parametrize("dt,n,m,bound", [("q8_0", 8037, 288, 6.4e-8), ("q8_0", 8000, 32, 6e-8),
                                          ("q4_0", 8000, 32, 9.5e-8), ("q4_0", 4096, 2880, 1.1e-7)])
def test_any_length_gemv_error(orc, dt, n, m, bound):
    """One token through the any-length GEMV is no further from 64 bits than the
    fp32 dot products of the any-shape kernel (bounds: what those measured, and
    sqrt(3.5) random roundings of 2.6e-8 for Q8_0, 4.9e-8, sqrt(8 to 14) for
    Q4_0, 7.5e-8 to 9.7e-8)."""
    import torch

    from hypno_amd import _lib
    print(f"{dt} n={n} m={m}", flush=True)
    rng = np.random.default_rng(n + m)
    w = (rng.standard_normal(n * m) * 0.02).astype(np.float32)
    wb = orc.quantize_q4_0(w) if dt == "q4_0" else orc.quantize_q8_0(w)
    x = rng.standard_normal((1, m)).astype(np.float32)
    got = _run(_lib.load(), torch, dt, wb, x, np.zeros(n, np.float32), n, m, 1, 0)
    f64 = orc.matmul_q4_0_f64 if dt == "q4_0" else orc.matmul_q8_0_f64
    assert orc.rel_l2(got[0], f64(wb, x[0], None, n, m)) <= bound


@pytest.mark.gpu
def test_any_shape_graph_outlives_larger_calls(orc):
    """A captured ragged batch replays right after calls that need a larger
    workspace on its stream."""
    import torch

    import hypno_amd as hk
    n, m, tokens = 2400, 2080, 17
    rng = np.random.default_rng(6)
    wb = orc.quantize_q4_0((rng.standard_normal(n * m) * 0.02).astype(np.float32))
    x = torch.from_numpy(rng.standard_normal((700, m)).astype(np.float32)).cuda()
    w = torch.from_numpy(wb).cuda()
    y, big = torch.zeros(tokens, n, device="cuda"), torch.zeros(700, n, device="cuda")
    s, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        hk.batch_matmul(y, w, hk.DType.Q4_0, x[:tokens], n, m, tokens)
    s.synchronize()
    want = y.clone()
    with torch.cuda.graph(g, stream=s):
        hk.batch_matmul(y, w, hk.DType.Q4_0, x[:tokens], n, m, tokens)
    for rows in (300, 700):
        with torch.cuda.stream(s):
            hk.batch_matmul(big[:rows], w, hk.DType.Q4_0, x[:rows], n, m, rows)
        s.synchronize()
        scratch = torch.full((1 << 24,), float("nan"), device="cuda")  # over freed memory
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
        del scratch
    for t in range(tokens):
        ref = orc.matmul_q4_0_f64(wb, x[t].cpu().numpy(), None, n, m)
        assert orc.normwise_err(want[t].cpu().numpy(), ref) <= 2e-5
