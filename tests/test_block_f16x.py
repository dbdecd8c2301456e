"""Prefill products on the block GEMM with x rounded once to fp16: Q8_0 from 16
tokens, and Q4_0 batches large enough for its 256-row tiles.  The cases sit one
row, column or K stage past its tiles (64, 128 and 256 rows, 256 columns, 64
columns of K), with and without K pieces; Q8_0 weights at an odd 2-byte address
take the expanded fp16 weights instead.

The reference multiplies the exact weights with x rounded as the kernels round
it, in 64 bits, so what is left is the fp32 sums.  An output passes through at
most K / 32 + 40 of their roundings (the blocks, the 32 products of one, K
pieces, scale and bias), each at most 2^-24 of a partial sum, which the sum of
the products' absolute values bounds."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu

CASES = [  # dtype, tokens, n, m
    ("q8_0", 16, 257, 64), ("q8_0", 17, 33, 128), ("q8_0", 33, 4096, 4096),
    ("q8_0", 64, 300, 2048), ("q8_0", 65, 1000, 320), ("q8_0", 127, 255, 8192),
    ("q8_0", 129, 513, 1088), ("q8_0", 257, 7201, 576), ("q8_0", 1025, 8193, 256),
    ("q8_0", 700, 1, 192), ("q8_0", 300, 1200, 16448), ("q8_0", 300, 16385, 512),
    ("q8_0", 128, 4097, 4160),
    ("q4_0", 1793, 5569, 1024), ("q4_0", 2048, 14336, 320), ("q4_0", 1025, 16385, 512),
    ("q4_0", 500, 14300, 2048), ("q4_0", 512, 14336, 64), ("q4_0", 1024, 16383, 64),
    ("q4_0", 2892, 2944, 3712),
]


def _blocks(torch, gen, n, m, dt):
    """Random blocks of n rows: their bytes and, in 64 bits, their values."""
    nb = n * m // 32
    d = (torch.rand(nb, generator=gen, device="cuda") * 0.02 + 1e-3).half()
    d[::7] *= -1
    size = 16 if dt == "q4_0" else 32
    q = torch.randint(0, 256, (nb, size), generator=gen, device="cuda", dtype=torch.uint8)
    w = torch.cat([d.view(torch.uint8).view(nb, 2), q], dim=1).contiguous().view(-1)
    if dt == "q4_0":
        v = torch.stack([q & 15, q >> 4], dim=2).view(nb, 32).double() - 8
    else:
        v = q.double() - 128
    return w, (v * d.double().unsqueeze(1)).view(n, m)


def _rounded(torch, x):
    """Rows scaled by the power of two that puts the largest |x| in
    [2^14, 2^15), rounded to fp16 and scaled back."""
    _, e = torch.frexp(x.abs().amax(dim=1, keepdim=True))
    return torch.ldexp(torch.ldexp(x, 15 - e).half().double(), e - 15)


def _run(torch, dt, w, x, bias, n, m, tokens):
    from hypno_amd import _lib
    lib = _lib.load()
    y = torch.full((tokens, n), float("nan"), device="cuda")
    fn = {"q4_0": lib.hypno_hip_matmul_q4_0_dev, "q8_0": lib.hypno_hip_matmul_q8_0_dev}[dt]
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    assert fn(p(y), p(w), w.numel(), p(x), p(bias), n, m, tokens, None) == 0
    torch.cuda.synchronize()
    return y


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("dt,tokens,n,m", CASES)
def test_block_f16x(dt, tokens, n, m, shift):
    import torch
    print(f"{dt} tokens={tokens} n={n} m={m} shift={shift}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(tokens * 31 + n + m)
    w, wv = _blocks(torch, gen, n, m, dt)
    buf = torch.randn(tokens * m + shift, generator=gen, device="cuda")
    x = buf[shift:].view(tokens, m)  # shifted: off a 16-byte boundary
    x[:, ::61] *= 30.0
    x[0] *= 1e-30
    if tokens > 20:
        x[19] = 0.0
    bias = torch.randn(n, generator=gen, device="cuda")
    got = _run(torch, dt, w, x, bias, n, m, tokens).double()
    xr = _rounded(torch, x)
    ref = xr @ wv.t() + bias.double()
    bound = (m / 32 + 40) * 2.0 ** -24 * (xr.abs() @ wv.abs().t() + bias.double().abs())
    bad = ((got - ref).abs() > bound) | got.isnan()
    assert not bad.any(), (bad.nonzero()[:4].tolist(), (got - ref).abs().max().item())


@pytest.mark.parametrize("tokens,n,m", [(40, 129, 320), (64, 300, 1088), (130, 300, 1088),
                                        (300, 5000, 1088)])
def test_q8_0_odd_address(tokens, n, m):
    """Weights at an odd 2-byte address: expanded to fp16, row by row scaled so
    that a block scale of 60000 (weights up to 127 * 60000) stays in range, on the
    streaming fp16 GEMM up to 64 tokens and the DMA-fed one beyond."""
    import torch
    gen = torch.Generator(device="cuda").manual_seed(3)
    w, wv = _blocks(torch, gen, n, m, "q8_0")
    big = torch.tensor([60000.0], dtype=torch.float16, device="cuda")
    blocks = w.view(n, m // 32, 34)
    for r, b in ((0, 0), (n - 1, m // 32 - 1)):
        blocks[r, b, :2] = big.view(torch.uint8)
        wv[r, 32 * b:32 * b + 32] = (blocks[r, b, 2:].double() - 128) * 60000.0
    buf = torch.empty(w.numel() + 2, dtype=torch.uint8, device="cuda")
    buf[2:] = w
    x = torch.randn(tokens, m, generator=gen, device="cuda")
    bias = torch.zeros(n, device="cuda")
    got = _run(torch, "q8_0", buf[2:], x, bias, n, m, tokens).double()
    ref = x.double() @ wv.t()
    # x and the weights each rounded to fp16 once: 2^-12 at random each
    for rows in (slice(1, n - 1), slice(0, 1), slice(n - 1, n)):
        g, r = got[:, rows], ref[:, rows]
        assert ((g - r).norm() / r.norm()).item() <= 1e-3
