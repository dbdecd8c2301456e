"""RMS norm over rows at the edges of the one-read kernel: widths around its
register tiles (1024, 2048 and 4096 vectors of 4), a last half vector pair
(n % 8 == 4), the element loop's widths and alignments beside it."""
import numpy as np
import pytest

EPS = 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("n,rows,shift", [(4, 3, 0), (12, 2, 0), (1020, 1, 0), (1024, 2, 0),
                                          (4096, 3, 0), (4100, 2, 0), (8192, 2, 0), (8196, 1, 0),
                                          (16384, 2, 0), (16388, 1, 0), (4095, 2, 0),
                                          (4096, 2, 1)])
def test_rms_norm_rows(orc, n, rows, shift):
    import torch

    import hypno_amd as hk
    rng = np.random.default_rng(n + rows)
    x = (rng.standard_normal(n * rows) * 3).astype(np.float32)
    w = (1.0 + 0.1 * rng.standard_normal(n)).astype(np.float32)
    ref = orc.rms_norm(x, w, EPS, rows)
    # shift: x starts 4 bytes past a 16-byte boundary
    dx = torch.empty(n * rows + shift, dtype=torch.float32, device="cuda")[shift:]
    dx.copy_(torch.from_numpy(x))
    dw = torch.from_numpy(w).cuda()
    got = hk.rms_norm(dx, dw, EPS, rows, out=torch.full_like(dx, float("nan")))
    hk.rms_norm_in_place(dx, dw, EPS, rows)
    torch.cuda.synchronize()
    g = got.cpu().numpy()
    assert np.array_equal(g, dx.cpu().numpy())
    # a sum of n squares in fp32 is within n * 2^-24 of exact in any order (far
    # less in this tree's); its root halves that; three roundings follow
    assert np.max(np.abs(g - ref)) / np.max(np.abs(ref)) <= 1e-5
